// adjoint.hip -- hand-written adjoint of shading and perspective-correct
// interpolation with visibility held fixed (no counterpart in the reference).
//
// For every covered pixel the winning input triangle comes from the forward
// pass's triangle-ID buffer; its vertices are re-read from the job's mesh and
// re-projected with the job's MVP.  The pixel's perspective-correct
// barycentrics are recomputed in continuous (unsnapped) clip space:
//   A_i = X_i - x W_i,  B_i = Y_i - y W_i,  q = A x B,  b = q / (q0 + q1 + q2)
// for the pixel centre (x, y) in NDC (the weights that put the clip-space
// point sum b_i c_i on the pixel's ray; the same weights Fragment::Interpolate,
// Core/Shader.h:142-170, forms from screen barycentrics and 1/w).  Using the
// input triangle, not a clipped piece, is exact: clipping is linear in clip
// space, so a clipped piece interpolates the same attributes.  The colour is
// the pixel shader of the forward pass (Core/Shader.h:209-282: diffuse =
// (max(N.L, 0) + ambient) kd / pi, spec = pow(N.H, s) ks) clamped to [0, 1];
// the adjoint back-propagates dL/dcolour to per-vertex positions (through
// shading and the barycentrics), normals, colours, the light direction and
// (ambient, kd, ks, shininess).
//
// Everything after the fp32 inputs is computed in double: a vertex's
// position gradient is the sum of many per-pixel terms that largely cancel
// (moving a vertex moves the barycentrics of every pixel of its triangles),
// so fp32 per-pixel arithmetic leaves relative errors of about 1e-3 at
// 512 x 512.  Per-vertex sums of a tile go to an LDS table keyed by vertex
// (double LDS atomics), then once per tile to the job's double accumulators,
// which a last pass adds to the float outputs.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pipeline.h"

namespace edxr {

namespace {

constexpr uint32_t kWave = 64;
constexpr uint32_t kAdjBlock = 256;  // threads per tile workgroup (each wave takes 4 of the 16 8x8 blocks)
constexpr double kInvPi = 1.0 / 3.14159265358979323846;

struct V3 {
    double x, y, z;
};
__device__ __forceinline__ V3 v3(double x, double y, double z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ V3 operator*(V3 a, double s) { return v3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ double dot(V3 a, V3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
// The gradients' multiply-adds may round once, for fewer double-precision
// instructions.  What decides whether and on which side of a kink a pixel
// contributes (an area of 0, a cosine of 0, a colour of 0 or 1) is computed
// operation by operation, from the vectors above on: with fused steps the area of
// coincident vertices and the cosine of light in the surface came out as rounding
// noise instead of 0.  (64 views at 512 x 512: backward 458 us with everything
// fused, 464 so, 478 with nothing fused.)
#pragma clang fp contract(fast)

// p[i] of device memory (a pointer read from memory would be loaded through as
// a generic one, which also counts against the LDS waits).
template <class T>
__device__ __forceinline__ T at(const T* p, size_t i) {
    return ((const __attribute__((address_space(1))) T*)p)[i];
}

struct F3 {
    float x, y, z;
};
__device__ __forceinline__ float opaque(float v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ V3 again(const F3& a) { return v3((double)opaque(a.x), (double)opaque(a.y), (double)opaque(a.z)); }
__device__ __forceinline__ double fused_dot(V3 a, V3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ V3 add_scaled(V3 a, V3 b, double s) { return v3(a.x + b.x * s, a.y + b.y * s, a.z + b.z * s); }
// d/dv of normalize(v) applied to the upstream gradient g (u = v / |v|).
__device__ __forceinline__ V3 normalize_back(V3 u, double invLen, V3 g) { return add_scaled(g, u, -fused_dot(u, g)) * invLen; }

__device__ __forceinline__ double pow_int(double x, int n) {
    double r = 1.0, b = x;
    unsigned u = (unsigned)n;
    while (u) {
        if (u & 1u) r *= b;
        u >>= 1;
        if (u) b *= b;
    }
    return r;
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

constexpr uint32_t kTilePixels = kTileSize * kTileSize;
// Per-tile vertex sums: 384 slots (a tile of triangles of ten pixels has about
// 60 vertices) keep three workgroups resident per CU; a vertex that finds no
// slot within kVertProbes goes straight to the accumulators.
constexpr uint32_t kVertSlots = 384, kVertProbes = 16;
constexpr uint32_t kVertSlotBits = 9;
static_assert(kVertSlots < 1u << kVertSlotBits, "a triangle's three slots and kVertSlots itself in 27 bits");
constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr uint32_t kVals = 9;    // gradients per vertex: position, normal, colour
constexpr uint32_t kAdjWaves = kAdjBlock / kWave;

// kPixels: the pixels of a tile that a workgroup takes.  At most one triangle
// per pixel, so the triangle table is never more than half full.
template <uint32_t kPixels>
struct AdjShared {
    static constexpr uint32_t kTriSlots = 2 * kPixels;
    double sum[kVertSlots * kVals];
    double wsum[kAdjWaves][8];
    uint32_t key[kVertSlots];
    uint32_t tri[kTriSlots];      // the tile's triangles,
    uint32_t count[kTriSlots];    // their pixels, then their first places, then their vertices' slots
    uint32_t list[kPixels];       // covered pixels by triangle: table entry << 10 | pixel
    uint16_t triUsed[kPixels];       // occupied entries of tri, and of key, in the order they were taken
    uint16_t used[kVertSlots];
    uint32_t nTri, nUsed;
    uint32_t waveSum[kAdjWaves];
};
static_assert(kTilePixels == 1u << 10, "AdjShared::list");

// Slot of vertex v in the tile's table (inserted if absent), or kVertSlots
// when kVertProbes slots are taken by others.
template <uint32_t kPixels>
__device__ __forceinline__ uint32_t vertex_slot(AdjShared<kPixels>& S, uint32_t v) {
    uint32_t h = __umulhi(v * 2654435761u, kVertSlots);
#pragma unroll 1
    for (uint32_t probe = 0; probe < kVertProbes; probe++) {
        const uint32_t k = S.key[h];
        if (k == v) return h;
        if (k == kEmpty) {
            const uint32_t old = atomicCAS(&S.key[h], kEmpty, v);
            if (old == kEmpty) S.used[atomicAdd(&S.nUsed, 1u)] = (uint16_t)h;
            if (old == kEmpty || old == v) return h;
        }
        if (++h == kVertSlots) h = 0;
    }
    return kVertSlots;
}

// Entry of triangle id in the tile's table (inserted if absent).
template <uint32_t kPixels>
__device__ __forceinline__ uint32_t tri_entry(AdjShared<kPixels>& S, uint32_t id) {
#pragma unroll 1
    for (uint32_t h = __umulhi(id * 2654435761u, 2 * kPixels);; h = (h + 1) & (2 * kPixels - 1)) {
        const uint32_t k = S.tri[h];
        if (k == id) return h;
        if (k == kEmpty) {
            const uint32_t old = atomicCAS(&S.tri[h], kEmpty, id);
            if (old == kEmpty) S.triUsed[atomicAdd(&S.nTri, 1u)] = (uint16_t)h;
            if (old == kEmpty || old == id) return h;
        }
    }
}

// v of the lane kShift below in the same row of 16 lanes (0 beyond the row).
template <int kShift>
__device__ __forceinline__ double row_below(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x110 + kShift, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x110 + kShift, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ uint32_t job_of(const BatchParams& Q, const uint32_t* tbl, uint32_t i) {
    return Q.num_jobs == 1 ? 0u : __builtin_amdgcn_readfirstlane(tbl[i]);
}

// A pixel's gradients before they are spread over its triangle's vertices:
// the interpolated attributes' (dP, dN, dC, vertex k taking b[k] of each) and
// those of the clip-space edge terms A, B (vertex k's position through the
// MVP), with the pixel centre in NDC.
struct PixelGrad {
    double b[3], dA[3], dB[3], xn, yn;
    V3 dP, dN, dC;
};

// The gradients of vertex k (position, normal, colour).
__device__ __forceinline__ void vertex_grad(const FrameParams& P, const PixelGrad& g, int k, double (&v)[kVals]) {
    const double b = g.b[k], dX = g.dA[k], dY = g.dB[k], dW = -g.xn * dX - g.yn * dY;
    const float* M = P.mvp;
    v[0] = g.dP.x * b + (((double)M[0] * dX + (double)M[4] * dY) + (double)M[12] * dW);
    v[1] = g.dP.y * b + (((double)M[1] * dX + (double)M[5] * dY) + (double)M[13] * dW);
    v[2] = g.dP.z * b + (((double)M[2] * dX + (double)M[6] * dY) + (double)M[14] * dW);
    v[3] = g.dN.x * b;
    v[4] = g.dN.y * b;
    v[5] = g.dN.z * b;
    v[6] = g.dC.x * b;
    v[7] = g.dC.y * b;
    v[8] = g.dC.z * b;
}

// The adjoint of one pixel: pg as above and the scalars gs[0..6] (light
// direction after normalisation, ambient, kd, ks, shininess).  Returns false
// for a pixel that contributes nothing.
// kPow: a job of the launch may have a shininess that is no whole exponent
// (pow is only compiled in then: its code and registers cost every job).
template <bool kPow>
__device__ __forceinline__ bool pixel_adjoint(const FrameParams& P, const uint32_t (&vi)[3], int x, int y,
                                              const float* gpix, PixelGrad& pg, double (&gs)[7]) {
    // The vertices are kept as the floats that they are and converted where
    // they are used (again(): not carried as doubles from one use to the
    // next), which holds the kernel to 168 VGPRs, three waves per SIMD.
    F3 pf[3], nf[3], cf[3];
    double A[3], Bc[3], xn, yn, q0, q1, q2, S;
    {
#pragma clang fp contract(off)
        double X[3], Y[3], W[3];
        const float* M = P.mvp;
        // the input vertices, read from the mesh (the forward stores shading
        // vertices only for vertices inside the frustum)
        const MeshPtrs& Mh = P.mesh;
        for (int k = 0; k < 3; k++) {
            const uint32_t v = vi[k];
            pf[k] = F3{at(Mh.px, v), at(Mh.py, v), at(Mh.pz, v)};
            nf[k] = F3{at(Mh.nx, v), at(Mh.ny, v), at(Mh.nz, v)};
            cf[k] = Mh.cr ? F3{at(Mh.cr, v), at(Mh.cg, v), at(Mh.cb, v)} : F3{0.0f, 0.0f, 0.0f};
            const V3 p = again(pf[k]);
            X[k] = (((double)M[0] * p.x + (double)M[1] * p.y) + (double)M[2] * p.z) + (double)M[3];
            Y[k] = (((double)M[4] * p.x + (double)M[5] * p.y) + (double)M[6] * p.z) + (double)M[7];
            W[k] = (((double)M[12] * p.x + (double)M[13] * p.y) + (double)M[14] * p.z) + (double)M[15];
        }
        // Pixel centre in NDC through the inverse of the raster matrix's 2D
        // affine part (x_r = R0 . (x, y) + R3, y_r likewise).
        const float* R = P.raster;
        const double r0 = R[0], r1 = R[1], r4 = R[4], r5 = R[5];
        const double rdet = r0 * r5 - r1 * r4;
        const double xr = (double)x + 0.5 - (double)R[3], yr = (double)y + 0.5 - (double)R[7];
        xn = (r5 * xr - r1 * yr) / rdet;
        yn = (r0 * yr - r4 * xr) / rdet;
        for (int k = 0; k < 3; k++) {
            A[k] = X[k] - xn * W[k];
            Bc[k] = Y[k] - yn * W[k];
        }
        q0 = A[1] * Bc[2] - A[2] * Bc[1];
        q1 = A[2] * Bc[0] - A[0] * Bc[2];
        q2 = A[0] * Bc[1] - A[1] * Bc[0];
        S = q0 + q1 + q2;
    }
    if (!(S != 0.0 && isfinite(S))) return false;
    const double invS = 1.0 / S;
    const double b[3] = {q0 * invS, q1 * invS, q2 * invS};
    pg.b[0] = b[0]; pg.b[1] = b[1]; pg.b[2] = b[2];
    pg.xn = xn; pg.yn = yn;
    const V3 Pw = (again(pf[0]) * b[0] + again(pf[1]) * b[1]) + again(pf[2]) * b[2];
    const V3 Nw = (again(nf[0]) * b[0] + again(nf[1]) * b[1]) + again(nf[2]) * b[2];
    const V3 Cw = (again(cf[0]) * b[0] + again(cf[1]) * b[1]) + again(cf[2]) * b[2];
    const double invN = rsqrt(dot(Nw, Nw));
    const V3 nh = Nw * invN;
    const V3 L = v3(P.light[0], P.light[1], P.light[2]);
    const double nl = dot(nh, L);
    const double dAmt = nl < 0.0 ? 0.0 : nl;
    const double ambient = P.ambient, kd = P.kd, ks = P.ks;
    const double diffuse = (dAmt + ambient) * kd * kInvPi;
    const bool lambert = P.shader == kLambertAlbedo;
    V3 base = P.shader == kVcBlinnPhong ? Cw : v3(1.0, 1.0, 1.0);
    if (lambert) base = v3(P.albedo[0], P.albedo[1], P.albedo[2]);
    double spec = 0.0, sa = 0.0, sk = 0.0, dsk = 0.0, invV = 0.0, invH = 0.0;
    V3 vh = v3(0, 0, 0), hh = v3(0, 0, 0);
    if (!lambert) {
        const V3 ev = v3(P.eye[0], P.eye[1], P.eye[2]) - Pw;
        invV = rsqrt(dot(ev, ev));
        vh = ev * invV;
        const V3 h = L + vh;
        invH = rsqrt(dot(h, h));
        hh = h * invH;
        sa = dot(nh, hh);
        if (P.clamp_spec) sa = fmax(sa, 0.0);
        if (!kPow || P.shin_int >= 0) {
            const double below = P.shin_int > 0 ? pow_int(sa, P.shin_int - 1) : 0.0;
            sk = P.shin_int > 0 ? below * sa : 1.0;
            dsk = (double)P.shin_int * below;
        } else {
            const double s = P.shininess;
            sk = pow(sa, s);
            dsk = s * pow(sa, s - 1.0);
        }
        spec = sk * ks;
    }
    double col[3];
    {
#pragma clang fp contract(off)
        col[0] = diffuse * base.x + spec;
        col[1] = diffuse * base.y + spec;
        col[2] = diffuse * base.z + spec;
    }
    double g[3];
    for (int ch = 0; ch < 3; ch++) {
        g[ch] = gpix[ch];
        if (!(col[ch] > 0.0 && col[ch] < 1.0)) g[ch] = 0.0;  // clamp
    }
    // colour = diffuse * base + spec
    const double dDiffuse = (g[0] * base.x + g[1] * base.y) + g[2] * base.z;
    const double dSpec = lambert ? 0.0 : (g[0] + g[1]) + g[2];
    const V3 dC = P.shader == kVcBlinnPhong ? v3(g[0] * diffuse, g[1] * diffuse, g[2] * diffuse) : v3(0.0, 0.0, 0.0);
    // diffuse = (max(n.L, 0) + ambient) kd / pi
    gs[3] = dDiffuse * kd * kInvPi;
    gs[4] = dDiffuse * (dAmt + ambient) * kInvPi;
    const double dnl = nl > 0.0 ? dDiffuse * kd * kInvPi : 0.0;
    V3 dnh = L * dnl;
    V3 dL = nh * dnl;
    V3 dP = v3(0.0, 0.0, 0.0);
    gs[5] = gs[6] = 0.0;
    if (!lambert) {
        // spec = pow(sa, s) ks
        gs[5] = dSpec * sk;
        gs[6] = sa > 0.0 ? dSpec * ks * sk * log(sa) : 0.0;
        double dsa = dSpec * ks * dsk;
        if (P.clamp_spec && !(dot(nh, hh) > 0.0)) dsa = 0.0;
        dnh = add_scaled(dnh, hh, dsa);
        const V3 dh = normalize_back(hh, invH, nh * dsa);  // h = L + v
        dL = dL + dh;
        dP = v3(0.0, 0.0, 0.0) - normalize_back(vh, invV, dh);  // v = normalize(eye - P)
    }
    gs[0] = dL.x;
    gs[1] = dL.y;
    gs[2] = dL.z;
    const V3 dN = normalize_back(nh, invN, dnh);
    // Interpolated attributes: d(attr_k) = b_k d(attr); d b_k = d(attr) . attr_k
    double db[3];
    pg.dP = dP; pg.dN = dN; pg.dC = dC;
    for (int k = 0; k < 3; k++) db[k] = (fused_dot(dP, again(pf[k])) + fused_dot(dN, again(nf[k]))) + fused_dot(dC, again(cf[k]));
    // b = q / S
    const double bdb = (b[0] * db[0] + b[1] * db[1]) + b[2] * db[2];
    const double dq[3] = {(db[0] - bdb) * invS, (db[1] - bdb) * invS, (db[2] - bdb) * invS};
    // q = A x B
    pg.dA[0] = Bc[1] * dq[2] - Bc[2] * dq[1];
    pg.dA[1] = Bc[2] * dq[0] - Bc[0] * dq[2];
    pg.dA[2] = Bc[0] * dq[1] - Bc[1] * dq[0];
    pg.dB[0] = A[2] * dq[1] - A[1] * dq[2];
    pg.dB[1] = A[0] * dq[2] - A[2] * dq[0];
    pg.dB[2] = A[1] * dq[0] - A[0] * dq[1];
    return true;
}

}  // namespace

__global__ void k_adjoint_zero(double* acc, uint64_t nacc, double* vacc, uint64_t n) {
    const uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, di = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = i0; i < nacc; i += di) acc[i] = 0.0;
    for (uint64_t i = i0; i < n; i += di) vacc[i] = 0.0;
}

// One workgroup per 32x32 tile.  Its covered pixels are first sorted by
// triangle in LDS (a counting sort over a table of the tile's triangles), so
// that only covered pixels take lanes and the pixels of a triangle are
// neighbours, and the vertices of each triangle get their slots in a table of
// sums.  Each wave then takes 64 pixels, one per lane: the 27 gradients of the
// lane's triangle's vertices are summed over the neighbouring lanes of the
// same triangle in registers (DPP row shifts), the last of them adds the sums
// to the table, and at the end the table's vertices are added to the
// accumulators.
// Adding every pixel's 27 values to the table with LDS atomics instead, where
// the lanes of a triangle meet on the same addresses and look up its vertices
// each, took 968 us for 64 views at 512 x 512 (3.8M covered pixels); this takes
// 353 us, bound by the latency of its double-precision chains at three waves
// per SIMD (168 VGPRs; about 1,200 vector instructions per 64 pixels).  Half
// a tile per workgroup takes 388 us, a quarter 468 us, two waves per SIMD
// without spills 425 us.
template <uint32_t kPixels, bool kPow>
__global__ __launch_bounds__(kAdjBlock, 3) void k_adjoint(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                          const GradPtrs* __restrict__ grads,
                                                          const uint32_t* __restrict__ ids,
                                                          const float* __restrict__ d_rgb, double* acc, double* vacc) {
    __shared__ AdjShared<kPixels> S;
    constexpr uint32_t kTriSlots = S.kTriSlots, kParts = kTilePixels / kPixels;
    const uint32_t gtile = blockIdx.x / kParts;
    const uint32_t job = job_of(Q, Q.tile_job, gtile);
    const FrameParams& P = jobs[job];
    const uint32_t tile = gtile - P.tile_base;
    // Rows of tiles are turned by three against each other: workgroups go to
    // the XCDs in turn, so that with 8, 16 or 32 tiles in a row every XCD
    // would have the same columns of every view, and those in the middle are
    // covered and those at the sides are not (64 views: 512 -> 368 us).
    const uint32_t row = tile / P.tiles_x;
    const int x0 = (int)((tile + 3 * row) % P.tiles_x) * kTileSize, y0 = (int)row * kTileSize + (int)(blockIdx.x % kParts * (kPixels / kTileSize));
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    constexpr uint32_t kPer = kPixels / kAdjBlock;
    auto offset_of = [&](uint32_t p) {
        const int x = x0 + (int)(p % kTileSize), y = y0 + (int)(p / kTileSize);
        return P.pix_base + (size_t)(P.height - 1 - y) * P.width + x;
    };
    uint32_t id[kPer];
    bool any = false;
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        const uint32_t p = threadIdx.x + u * kAdjBlock;
        const bool inside = x0 + (int)(p % kTileSize) < (int)P.width && y0 + (int)(p / kTileSize) < (int)P.height;
        id[u] = inside ? ids[offset_of(p)] : kEmpty;
        any |= id[u] != kEmpty;
    }
    if (!__syncthreads_or(any)) return;  // nothing covered
    for (uint32_t i = threadIdx.x; i < kTriSlots; i += kAdjBlock) {
        S.tri[i] = kEmpty;
        S.count[i] = 0;
    }
    for (uint32_t i = threadIdx.x; i < kVertSlots; i += kAdjBlock) S.key[i] = kEmpty;
    for (uint32_t i = threadIdx.x; i < kVertSlots * kVals; i += kAdjBlock) S.sum[i] = 0.0;
    if (threadIdx.x == 0) S.nUsed = S.nTri = 0;
    __syncthreads();
    // The counting sort: each pixel's place among its triangle's, the
    // triangles' first places, the list.
    uint32_t entry[kPer], rank[kPer];
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        if (id[u] == kEmpty) continue;
        entry[u] = tri_entry(S, id[u]);
        rank[u] = atomicAdd(&S.count[entry[u]], 1u);
    }
    __syncthreads();
    // (the scan in the order of the entries: kPerScan neighbours per thread)
    constexpr uint32_t kPerScan = kTriSlots / kAdjBlock;
    uint32_t own = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPerScan; u++) own += S.count[threadIdx.x * kPerScan + u];
    uint32_t incl = own;
    for (uint32_t o = 1; o < kWave; o <<= 1) {
        const uint32_t v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    if (lane == kWave - 1) S.waveSum[wave] = incl;
    __syncthreads();
    uint32_t total = 0, run = incl - own;
    for (uint32_t w = 0; w < kAdjWaves; w++) {
        if (w < wave) run += S.waveSum[w];
        total += S.waveSum[w];
    }
#pragma unroll
    for (uint32_t u = 0; u < kPerScan; u++) {
        const uint32_t c = S.count[threadIdx.x * kPerScan + u];
        S.count[threadIdx.x * kPerScan + u] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++)
        if (id[u] != kEmpty)
            S.list[S.count[entry[u]] + rank[u]] = entry[u] << 10 | (threadIdx.x + u * kAdjBlock);
    __syncthreads();  // the places are read: count takes the vertices' slots
    for (uint32_t i = threadIdx.x; i < S.nTri; i += kAdjBlock) {
        const uint32_t e = S.triUsed[i];
        const size_t t = 3 * (size_t)S.tri[e];
        const uint32_t v0 = at(P.mesh.idx, t), v1 = at(P.mesh.idx, t + 1), v2 = at(P.mesh.idx, t + 2);
        S.count[e] = vertex_slot(S, v0) | vertex_slot(S, v1) << kVertSlotBits | vertex_slot(S, v2) << 2 * kVertSlotBits;
    }
    __syncthreads();

    const GradPtrs& G = grads[job];
    double gsum[7] = {0, 0, 0, 0, 0, 0, 0};
    // (the next pixels' indices are loaded before this step's work)
    auto fetch = [&](uint32_t base, uint32_t& item, uint32_t (&vi)[3]) {
        item = S.list[min(base + lane, total - 1)];
        const size_t i = 3 * (size_t)S.tri[item >> 10];
#pragma unroll
        for (int k = 0; k < 3; k++) vi[k] = at(P.mesh.idx, i + k);
    };
    uint32_t next, nextVi[3];
    if (wave * kWave < total) fetch(wave * kWave, next, nextVi);
    for (uint32_t base = wave * kWave; base < total; base += kAdjBlock) {
        const bool live = base + lane < total;
        const uint32_t e = next >> 10, p = next & (kTilePixels - 1), vi[3] = {nextVi[0], nextVi[1], nextVi[2]};
        if (base + kAdjBlock < total) fetch(base + kAdjBlock, next, nextVi);
        PixelGrad pg;
        double gs[7];
        const bool ok = live && pixel_adjoint<kPow>(P, vi, x0 + (int)(p % kTileSize), y0 + (int)(p / kTileSize),
                                              d_rgb + 3 * offset_of(p), pg, gs);
        if (ok) {
#pragma unroll
            for (int j = 0; j < 7; j++) gsum[j] += gs[j];
        }
        // Runs: a triangle's pixels in neighbouring lanes of a half row.  A
        // lane adds the lanes 1, 2 and 4 below while they are of its run.
        const uint32_t run = live ? e : kTriSlots + lane;  // (a lane without a pixel is a run of its own)
        const uint32_t sub = lane & 7u;
        const uint32_t b1 = __shfl_up(run, 1), b2 = __shfl_up(run, 2), b4 = __shfl_up(run, 4);
        const bool add1 = sub >= 1 && b1 == run, add2 = sub >= 2 && b2 == run, add4 = sub >= 4 && b4 == run;
        const uint32_t above = __shfl_down(run, 1);
        const bool last = live && (sub == 7 || above != run);
        const uint32_t slots = S.count[e];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            double v[kVals];
            vertex_grad(P, pg, k, v);
            const uint32_t vs = (slots >> (k * kVertSlotBits)) & ((1u << kVertSlotBits) - 1);
#pragma unroll
            for (uint32_t j = 0; j < kVals; j++) {
                double t = ok ? v[j] : 0.0;
                const double t1 = row_below<1>(t);
                t += add1 ? t1 : 0.0;
                const double t2 = row_below<2>(t);
                t += add2 ? t2 : 0.0;
                const double t4 = row_below<4>(t);
                t += add4 ? t4 : 0.0;
                v[j] = t;
            }
            if (last && vs < kVertSlots) {
#pragma unroll
                for (uint32_t j = 0; j < kVals; j++) atomicAdd(&S.sum[vs * kVals + j], v[j]);
            } else if (last) {
#pragma unroll
                for (uint32_t j = 0; j < kVals; j++)
                    atomicAdd(&vacc[G.acc_base + (uint64_t)vi[k] * kVals + j], v[j]);
            }
        }
    }
    // Scalars: wave sums, then one double atomic per workgroup and value.
#pragma unroll
    for (int j = 0; j < 7; j++) {
        const double s = wave_sum(gsum[j]);
        if (lane == 0) S.wsum[wave][j] = s;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        double t = 0.0;
        for (uint32_t w = 0; w < kAdjWaves; w++) t += S.wsum[w][threadIdx.x];
        if (t != 0.0) atomicAdd(&acc[8 * job + threadIdx.x], t);
    }
    for (uint32_t w = threadIdx.x; w < S.nUsed * kVals; w += kAdjBlock) {
        const uint32_t vs = S.used[w / kVals], j = w % kVals;
        const double t = S.sum[vs * kVals + j];
        if (t != 0.0) atomicAdd(&vacc[G.acc_base + (uint64_t)S.key[vs] * kVals + j], t);
    }
}

// The caller's arrays.  The first workgroups take 64 jobs each: the jobs'
// light gradients through Normalize (L = l / |l|) and material gradients; jobs
// of one wave that share their outputs (the usual case: views of one scene)
// are summed in double first, since atomics of 64 jobs on seven addresses
// queue up.  The others take parts of a job each: every part of the first job
// of a group sharing vertex outputs adds its share of the group's double
// accumulators (vertex-major), rounded once.  (One workgroup per group, after
// a launch for the scalars: 144 + 9 us for 64 views of 10,000 vertices; this
// takes 15 us.)
__global__ __launch_bounds__(256) void k_adjoint_finish(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                        const GradPtrs* __restrict__ grads, const double* acc,
                                                        const double* vacc, uint32_t scalarBlocks) {
    if (blockIdx.x < scalarBlocks) {
        const uint32_t job = blockIdx.x * kWave + threadIdx.x;
        if (threadIdx.x >= kWave) return;
        const bool live = job < Q.num_jobs;
        const FrameParams& P = jobs[live ? job : 0u];
        const GradPtrs& G = grads[live ? job : 0u];
        double v[7];
        for (int k = 0; k < 7; k++) v[k] = live ? acc[8 * job + k] : 0.0;
        const double L[3] = {P.light[0], P.light[1], P.light[2]};
        const double LdL = L[0] * v[0] + L[1] * v[1] + L[2] * v[2];
        for (int k = 0; k < 3; k++) v[k] = (v[k] - L[k] * LdL) / (double)P.light_len;
        const GradPtrs& F = grads[blockIdx.x * kWave];  // the wave's first job
        if (__ballot(live && (G.d_light != F.d_light || G.d_material != F.d_material)) == 0) {
            for (int k = 0; k < 7; k++) v[k] = wave_sum(live ? v[k] : 0.0);
            if (threadIdx.x != 0) return;
        }
        if (!live) return;
        if (G.d_light)
            for (int k = 0; k < 3; k++) atomicAdd(&G.d_light[k], (float)v[k]);
        if (G.d_material)
            for (int k = 0; k < 4; k++) atomicAdd(&G.d_material[k], (float)v[3 + k]);
        return;
    }
    const uint32_t b = blockIdx.x - scalarBlocks, job = b % Q.num_jobs, part = b / Q.num_jobs;
    const uint32_t parts = (gridDim.x - scalarBlocks) / Q.num_jobs;
    const GradPtrs& G = grads[job];
    if (!G.group_first) return;
    float* const outs[kVals] = {G.d_px, G.d_py, G.d_pz, G.d_nx, G.d_ny, G.d_nz, G.d_cr, G.d_cg, G.d_cb};
    for (uint32_t v = part * 256 + threadIdx.x; v < G.acc_v; v += parts * 256) {
        const double* a = vacc + G.acc_base + (uint64_t)v * kVals;
#pragma unroll
        for (uint32_t j = 0; j < kVals; j++)
            if (outs[j] && a[j] != 0.0) atomicAdd(outs[j] + v, (float)a[j]);
    }
}

// Up to this many tiles, which leave resident workgroups idle (three per CU),
// four workgroups share a tile, so that a wave has one step instead of four:
// 196 tiles 43 -> 17 us; 16,384 tiles 359 -> 468 us.
constexpr uint32_t kSplitTiles = 768;

hipError_t launch_adjoint(const BatchParams& Q, const FrameParams* jobs, const GradPtrs* grads,
                          const uint32_t* ids, const float* d_rgb, double* acc,
                          double* vacc, uint64_t vacc_size, bool any_pow, hipStream_t s) {
    const uint64_t nacc = 8ull * Q.num_jobs;
    hipLaunchKernelGGL(k_adjoint_zero, dim3((uint32_t)std::min<uint64_t>((nacc + vacc_size + 255) / 256, 2048)),
                       dim3(256), 0, s, acc, nacc, vacc, vacc_size);
    auto launch = [&](auto kernel, uint32_t parts) {
        hipLaunchKernelGGL(kernel, dim3(parts * Q.total_tiles), dim3(kAdjBlock), 0, s, Q, jobs, grads, ids, d_rgb, acc,
                           vacc);
    };
    if (Q.total_tiles && Q.total_tiles <= kSplitTiles) {
        if (any_pow) launch(k_adjoint<kTilePixels / 4, true>, 4);
        else launch(k_adjoint<kTilePixels / 4, false>, 4);
    } else if (Q.total_tiles) {
        if (any_pow) launch(k_adjoint<kTilePixels, true>, 1);
        else launch(k_adjoint<kTilePixels, false>, 1);
    }
    // parts per job: enough for a vertex per thread of the largest possible
    // group, and no more than 4096 workgroups beyond one per job
    const uint64_t want = (vacc_size / kVals + 255) / 256;
    const uint32_t parts = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(want, 4096 / Q.num_jobs));
    const uint32_t scalarBlocks = (Q.num_jobs + kWave - 1) / kWave;
    hipLaunchKernelGGL(k_adjoint_finish, dim3(scalarBlocks + Q.num_jobs * parts), dim3(256), 0, s, Q, jobs, grads, acc,
                       vacc, scalarBlocks);
    return hipGetLastError();
}

}  // namespace edxr
