// ds.hip -- GatherDistGrad (src/core/f_ops.cpp:1248-1358): the exact
// backward of RasterizeSoft's dist channel w.r.t. the hard clip positions
// (the backward RasterizeSoft builds, f_ops.cpp:1448-1455, and what
// dressi.torch.rasterize_soft's VJP runs).
#include <algorithm>
#include <cstdint>

#include "internal.h"
#include "soft_clip.h"
#include "surface_core.h"

namespace dressi {
namespace {

// cpu_raster.cpp:114-151 (SignedDistToTri) with the argmin edge, its clamped
// parameter and its nearest point (kept here: found again from the edge's
// run-time index it would put the corner arrays in scratch).
struct TriDistE {
    float dist;
    int edge;
    float t;
    float qx, qy;
};

__device__ __forceinline__ TriDistE signed_dist_edge(float px, float py, const float sx[3],
                                                     const float sy[3]) {
    TriDistE best;
    best.dist = 0.f;
    best.edge = 0;
    best.t = 0.f;
    best.qx = best.qy = 0.f;
    float best_d2 = -1.f;
    int n_pos = 0, n_neg = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int k1 = (k + 1) % 3;
        const float ex = sx[k1] - sx[k];
        const float ey = sy[k1] - sy[k];
        const float len2 = ex * ex + ey * ey;
        float t = 0.f;
        if (len2 > kDistEps * kDistEps) {
            t = ((px - sx[k]) * ex + (py - sy[k]) * ey) / len2;
            t = smin(smax(t, 0.f), 1.f);
        }
        const float qx = sx[k] + t * ex;
        const float qy = sy[k] + t * ey;
        const float dx = px - qx;
        const float dy = py - qy;
        const float d2 = dx * dx + dy * dy;
        if (best_d2 < 0.f || d2 < best_d2) {
            best_d2 = d2;
            best.edge = k;
            best.t = t;
            best.qx = qx;
            best.qy = qy;
        }
        const float cr = ex * (py - sy[k]) - ey * (px - sx[k]);
        n_pos += (cr >= 0.f);
        n_neg += (cr <= 0.f);
    }
    const float sgn = (n_pos == 3 || n_neg == 3) ? 1.f : -1.f;
    best.dist = sgn * sqrtf(smax(best_d2, 0.f));
    return best;
}

// cpu_raster.cpp:153-175 (SignedDistGradToTri): d dist / d corner k, the
// argmin edge and t held fixed (envelope theorem); 0 on the boundary.
__device__ __forceinline__ void signed_dist_grad_k(float px, float py, const float sx[3],
                                                   const float sy[3], const TriDistE& td, int k,
                                                   float* gx, float* gy) {
    *gx = 0.f;
    *gy = 0.f;
    const float d = fabsf(td.dist);
    if (d < kDistEps) {
        return;
    }
    const int ia = td.edge;
    const int ib = (td.edge + 1) % 3;
    if (k != ia && k != ib) {
        return;
    }
    const float sgn = td.dist >= 0.f ? 1.f : -1.f;
    const float nx = (px - td.qx) / d;
    const float ny = (py - td.qy) / d;
    if (k == ia) {
        *gx = -sgn * (1.f - td.t) * nx;
        *gy = -sgn * (1.f - td.t) * ny;
    } else {
        *gx = -sgn * td.t * nx;
        *gy = -sgn * td.t * ny;
    }
}

// A face's corners: vertex ids, hard clips and projected screen positions;
// false when a corner is not projectable (the reference skips its pixels).
struct FaceCorners {
    uint32_t idx[3];
    float4 c[3];
    float sx[3], sy[3];
};

__device__ __forceinline__ bool load_face(const float* faces, const float4* clip, uint32_t n_verts,
                                          uint32_t f, float W, float H, FaceCorners* fc,
                                          uint32_t* err) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        fc->idx[k] = (uint32_t)(int64_t)(faces[(size_t)f * 3 + k] + 0.5f);
        if (fc->idx[k] >= n_verts) {
            atomicOr(err, 2u);
            return false;
        }
        fc->c[k] = clip[fc->idx[k]];
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (!clip_w_valid(fc->c[k].w)) {
            return false;
        }
        const ScreenVert v = project_to_screen(fc->c[k].x, fc->c[k].y, fc->c[k].z, fc->c[k].w, W, H);
        fc->sx[k] = v.x;
        fc->sy[k] = v.y;
    }
    return true;
}

// The pixel bbox of a face's soft triangle (SoftClip of its hard clips, as
// the soft raster's setup): every pixel whose RasterizeSoft winner is the
// face lies in it. False when the face produces no fragment.
__device__ __forceinline__ bool soft_bbox(const FaceCorners& fc, uint32_t w, uint32_t h,
                                          float radius, int* bx0, int* by0, int* bx1, int* by1) {
    float4 sc[3];
    soft_clip_face(fc.c, w, h, radius, sc);
    float x[3], y[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (!clip_w_valid(sc[k].w)) {
            return false;
        }
        const ScreenVert v = project_to_screen(sc[k].x, sc[k].y, sc[k].z, sc[k].w, (float)w, (float)h);
        x[k] = v.x;
        y[k] = v.y;
    }
    if (fabsf(tri_area(x[0], y[0], x[1], y[1], x[2], y[2])) < kDistEps) {
        return false;
    }
    pixel_bbox(x[0], x[1], x[2], y[0], y[1], y[2], (int)w, (int)h, bx0, by0, bx1, by1);
    return *bx0 <= *bx1 && *by0 <= *by1;
}

// Adds pixel (x, y)'s contribution to corner k of `fc` into acc (the
// screen -> clip Jacobian of f_ops.cpp:1342-1350).
__device__ __forceinline__ void add_corner(const FaceCorners& fc, const TriDistE& td, float px,
                                           float py, int k, float g, float W, float H,
                                           float4* acc) {
    float gsx0, gsy0;
    signed_dist_grad_k(px, py, fc.sx, fc.sy, td, k, &gsx0, &gsy0);
    const float gsx = g * gsx0;
    const float gsy = g * gsy0;
    if (gsx == 0.f && gsy == 0.f) {
        return;
    }
    const float4 c = fc.c[k];
    acc->x += gsx * 0.5f * W / c.w;
    acc->y += gsy * 0.5f * H / c.w;
    acc->w += -(gsx * 0.5f * W * c.x + gsy * 0.5f * H * c.y) / (c.w * c.w);
}

// Wide layout, row (d, u): face f = vtx_faces[d][u]'s pixels in raster order
// (its soft bbox, face-id guard), the corners that are u; only the first row
// holding f for u receives (the reference's row_of). Two kernels: every row
// cleared and its indices checked, then one wave per face that adds its
// pixels' contributions into its corners' rows.
//
// One thread per row scanned its face's box alone: each face three times,
// one pixel after another at a memory latency each, and the last threads'
// boxes (edge-on faces, up to 12 k pixels) set the time: 3.8 ms at 512 x 512,
// 5120 faces. The wave looks at 8 x 64 pixels at once and keeps the few that
// the face won (at most ~250 here); these are evaluated side by side, and
// only the adds go one by one: 56 us, set by the largest boxes' steps at a
// memory latency each (124 us when each step's hits were evaluated at once;
// four waves to a face 93 us: the setup's divisions repeat per wave).
__global__ __launch_bounds__(256) void k_gather_dist_grad_rows(const float* faces, uint32_t n_verts,
                                                               uint32_t n_faces, const float* vf,
                                                               uint32_t max_deg, uint32_t* err,
                                                               float4* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= max_deg * n_verts) {
        return;
    }
    const float fv = vf[i];
    out[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (fv >= -0.5f) {
        const uint32_t f = (uint32_t)(int64_t)(fv + 0.5f);
        bool ok = f < n_faces;
        for (int k = 0; k < 3 && ok; k++) {
            ok = (uint32_t)(int64_t)(faces[(size_t)f * 3 + k] + 0.5f) < n_verts;
        }
        if (!ok) {
            atomicOr(err, 2u);
        }
    }
}

// Pixels per lane and step (loads in flight); pixels that the face won kept
// before they are evaluated.
constexpr uint32_t kDistPx = 8;
constexpr uint32_t kDistHits = 1024;
static_assert(kDistHits >= 2 * 64 * kDistPx, "a step's hits fit beside those kept");

struct DistLds {
    uint32_t hit_px[kDistHits];
    float term[64][9];  // per hit: corner k's x, y, w contributions
};

// The sum of one face's pixels' contributions by one wave, in raster order:
// lane 3 r + c < 9 gets component c (x, y, w) of corner r's row. rs and gy are
// the item's images.
__device__ __forceinline__ float dist_face_sum(const FaceCorners& fc, uint32_t f, int bx0, int by0,
                                               uint32_t bw, uint32_t n_px, const float4* rs,
                                               const float4* gy, uint32_t w, float W, float H,
                                               DistLds& lds) {
    const uint32_t lane = threadIdx.x;
    const uint32_t r = lane < 9 ? lane / 3 : 0, comp = lane < 9 ? lane % 3 : 0;
    const uint32_t my = r == 0 ? fc.idx[0] : r == 1 ? fc.idx[1] : fc.idx[2];
    const bool twice = fc.idx[0] == fc.idx[1] || fc.idx[1] == fc.idx[2] || fc.idx[2] == fc.idx[0];
    float acc = 0.f;
    uint32_t n_hits = 0;
    const uint32_t origin = (uint32_t)by0 * w + (uint32_t)bx0;
    BoxWalk at((uint32_t)bx0, (uint32_t)by0, bw, w, lane);
    for (uint32_t p0 = 0; p0 < n_px; p0 += 64 * kDistPx) {
        uint32_t o[kDistPx];
        float2 yw[kDistPx];  // the winner's face id, coverage
#pragma unroll
        for (uint32_t s = 0; s < kDistPx; s++) {
            const bool in = p0 + s * 64 + lane < n_px;
            o[s] = in ? at.o : origin;
            at.next();
            const float4 v = rs[o[s]];
            yw[s] = make_float2(v.y, in ? v.w : 0.f);
        }
#pragma unroll
        for (uint32_t s = 0; s < kDistPx; s++) {
            const bool hit = !(yw[s].y < 0.5f) && (uint32_t)(int64_t)(yw[s].x + 0.5f) == f;
            const uint64_t m = __ballot(hit);
            if (hit) {
                lds.hit_px[n_hits + __popcll(m & ((1ull << lane) - 1ull))] = o[s];
            }
            n_hits += (uint32_t)__popcll(m);
        }
        const bool last = p0 + 64 * kDistPx >= n_px;
        if (!last && n_hits + 64 * kDistPx <= kDistHits) {
            continue;
        }
        wave_lds_fence();
        for (uint32_t h0 = 0; h0 < n_hits; h0 += 64) {
            const uint32_t n = min(64u, n_hits - h0);
            if (lane < n) {
                const uint32_t px_o = lds.hit_px[h0 + lane];
                const uint32_t y = px_o / w, x = px_o - y * w;
                const float g = gy[px_o].x;
                float4 t[3] = {};
                if (g != 0.f) {
                    const float px = (float)x + 0.5f, py = (float)y + 0.5f;
                    const TriDistE td = signed_dist_edge(px, py, fc.sx, fc.sy);
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        add_corner(fc, td, px, py, k, g, W, H, &t[k]);
                    }
                }
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    lds.term[lane][k * 3 + 0] = t[k].x;
                    lds.term[lane][k * 3 + 1] = t[k].y;
                    lds.term[lane][k * 3 + 2] = t[k].w;
                }
            }
            wave_lds_fence();
            // a contribution that the reference leaves out is +0 here: a sum
            // that starts at +0 is never -0, and +0 leaves it as it is
            if (lane < 9 && !twice) {
#pragma unroll 8
                for (uint32_t q = 0; q < n; q++) {
                    acc += lds.term[q][lane];
                }
            } else if (lane < 9) {
                for (uint32_t q = 0; q < n; q++) {
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        if (fc.idx[k] == my) {
                            acc += lds.term[q][k * 3 + comp];
                        }
                    }
                }
            }
            wave_lds_fence();
        }
        n_hits = 0;
    }
    return acc;
}

// dist_face_sum's sums into the rows of face f's corners: of each vertex's rows
// the first that holds f.
__device__ __forceinline__ void dist_write_rows(const FaceCorners& fc, uint32_t f, float acc,
                                                const float* vf, uint32_t n_verts,
                                                uint32_t max_deg, float4* out) {
    const uint32_t lane = threadIdx.x;
    const uint32_t r = lane < 9 ? lane / 3 : 0, comp = lane < 9 ? lane % 3 : 0;
    const uint32_t my = r == 0 ? fc.idx[0] : r == 1 ? fc.idx[1] : fc.idx[2];
    uint32_t row = max_deg;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        uint32_t at = max_deg;
        for (uint32_t d0 = 0; d0 < max_deg && at == max_deg; d0 += 64) {
            const uint32_t d = d0 + lane;
            const float fv = d < max_deg ? vf[(size_t)d * n_verts + fc.idx[k]] : -1.f;
            const uint64_t m = __ballot(fv >= -0.5f && (uint32_t)(int64_t)(fv + 0.5f) == f);
            if (m) {
                at = d0 + (uint32_t)__builtin_ctzll(m);
            }
        }
        row = (int)r == k ? at : row;
    }
    if (lane < 9 && row < max_deg) {
        float* dst = (float*)&out[(size_t)row * n_verts + my];
        dst[comp == 2 ? 3 : comp] = acc;
    }
}

__global__ __launch_bounds__(64) void k_gather_dist_grad_faces(
        const float4* gy, const float4* rs, const float4* clip, uint32_t n_verts,
        const float* faces, const float* vf, uint32_t max_deg, float radius, uint32_t w,
        uint32_t h, float4* out) {
    __shared__ DistLds lds;
    const uint32_t f = blockIdx.x, lane = threadIdx.x;
    const float W = (float)w, H = (float)h;
    // (bad indices are the row kernel's to report)
    for (int k = 0; k < 3; k++) {
        if ((uint32_t)(int64_t)(faces[(size_t)f * 3 + k] + 0.5f) >= n_verts) {
            return;
        }
    }
    FaceCorners fc;
    int bx0, by0, bx1, by1;
    if (!load_face(faces, clip, n_verts, f, W, H, &fc, nullptr) ||
        !soft_bbox(fc, w, h, radius, &bx0, &by0, &bx1, &by1)) {
        return;
    }
    const uint32_t bw = (uint32_t)(bx1 - bx0 + 1);
    const uint32_t n_px = bw * (uint32_t)(by1 - by0 + 1);
    const float acc = dist_face_sum(fc, f, bx0, by0, bw, n_px, rs, gy, w, W, H, lds);
    dist_write_rows(fc, f, acc, vf, n_verts, max_deg, out);
}

// The torch surface's form: every item and peel, corner sums {N,K,F,3}
// (x, y, w) for an adjacency of the same faces. A wave per face, item and
// peel: what bounds is its chain of loads, and two peels in one wave after
// one setup took 115 us for two 512 x 512 views of 5120 faces, side by side
// 87.
__global__ __launch_bounds__(64) void k_surface_soft_bwd_faces(
        const float4* gy, const float4* rs, uint32_t peels, const float4* pos, uint32_t n_verts,
        const float* faces, uint32_t n_faces, float radius, uint32_t w, uint32_t h,
        float* g_corner) {
    __shared__ DistLds lds;
    const uint32_t f = blockIdx.x, lane = threadIdx.x;
    const float W = (float)w, H = (float)h;
    const size_t npx = (size_t)w * h;
    pos += (size_t)blockIdx.y * n_verts;
    bool ok = true;
    for (int k = 0; k < 3; k++) {
        ok = ok && fid_u(faces[(size_t)f * 3 + k]) < n_verts;
    }
    FaceCorners fc;
    int bx0 = 1, by0 = 1, bx1 = 0, by1 = 0;
    ok = ok && load_face(faces, pos, n_verts, f, W, H, &fc, nullptr) &&
         soft_bbox(fc, w, h, radius, &bx0, &by0, &bx1, &by1);
    const uint32_t bw = (uint32_t)(bx1 - bx0 + 1);
    const uint32_t n_px = ok ? bw * (uint32_t)(by1 - by0 + 1) : 0u;
    for (uint32_t k = blockIdx.z; k < peels; k += gridDim.z) {
        const size_t layer = (size_t)blockIdx.y * peels + k;
        float acc = 0.f;
        if (n_px) {
            acc = dist_face_sum(fc, f, bx0, by0, bw, n_px, rs + layer * npx, gy + layer * npx, w,
                                W, H, lds);
        }
        if (lane < 9) {
            g_corner[(layer * n_faces + f) * 9 + lane] = acc;
        }
    }
}

// Face f's corners and soft box; 0 pixels for a face that wins none.
__device__ __forceinline__ uint32_t dist_face(const float* faces, const float4* clip,
                                              uint32_t n_verts, uint32_t f, float radius,
                                              uint32_t w, uint32_t h, FaceCorners* fc, int* bx0,
                                              int* by0, uint32_t* bw) {
    bool ok = true;
    for (int k = 0; k < 3; k++) {
        ok = ok && fid_u(faces[(size_t)f * 3 + k]) < n_verts;
    }
    int bx1, by1;
    if (!ok || !load_face(faces, clip, n_verts, f, (float)w, (float)h, fc, nullptr) ||
        !soft_bbox(*fc, w, h, radius, bx0, by0, &bx1, &by1)) {
        return 0;
    }
    *bw = (uint32_t)(bx1 - *bx0 + 1);
    return *bw * (uint32_t)(by1 - *by0 + 1);
}

// Faces whose boxes are too large for a lane of k_dist_lanes.
struct DistBig {
    uint32_t* n;  // zero before
    uint2* list;  // (face, layer), room for all
};

// The listed faces, a wave at a time.
template <bool ROWS>
__global__ __launch_bounds__(64, 6) void k_dist_big(
        const float4* gy, const float4* rs, uint32_t peels, const float4* clip, uint32_t n_verts,
        const float* faces, uint32_t n_faces, const float* vf, uint32_t max_deg, float radius,
        uint32_t w, uint32_t h, DistBig bigs, float* g_corner, float4* out) {
    __shared__ DistLds lds;
    const size_t npx = (size_t)w * h;
    const uint32_t n = *bigs.n;
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const uint2 e = bigs.list[i];
        const float4* c = clip + (size_t)(e.y / peels) * n_verts;
        FaceCorners fc;
        int x0, y0;
        uint32_t bw;
        const uint32_t n_px = dist_face(faces, c, n_verts, e.x, radius, w, h, &fc, &x0, &y0, &bw);
        const float acc = dist_face_sum(fc, e.x, x0, y0, bw, n_px, rs + e.y * npx, gy + e.y * npx,
                                        w, (float)w, (float)h, lds);
        if (ROWS) {
            dist_write_rows(fc, e.x, acc, vf, n_verts, max_deg, out);
        } else if (threadIdx.x < 9) {
            g_corner[((size_t)e.y * n_faces + e.x) * 9 + threadIdx.x] = acc;
        }
    }
}

// Both forms for many small faces, a lane per face: lanes go through their own
// boxes of up to kDistLaneBox pixels and list the few that the face won, and
// evaluate them together; larger boxes are k_dist_big's.
// ROWS: the wide layout's rows, else g_corner of every item and peel.
constexpr uint32_t kDistLaneBox = 256;
constexpr uint32_t kDistLaneHits = kDistHits / 64;
static_assert(kDistLaneHits >= 2 * kDistPx, "a step's hits fit beside those kept");

template <bool ROWS>
__global__ __launch_bounds__(64) void k_dist_lanes(
        const float4* gy, const float4* rs, uint32_t peels, const float4* clip, uint32_t n_verts,
        const float* faces, uint32_t n_faces, const float* vf, uint32_t max_deg, float radius,
        uint32_t w, uint32_t h, DistBig bigs, float* g_corner, float4* out) {
    __shared__ DistLds lds;
    const uint32_t lane = threadIdx.x, f = blockIdx.x * 64 + lane;
    const float W = (float)w, H = (float)h;
    const size_t npx = (size_t)w * h;
    clip += (size_t)blockIdx.y * n_verts;
    FaceCorners fc;
    int bx0 = 0, by0 = 0;
    uint32_t bw = 1;
    const uint32_t n_box =
            f < n_faces ? dist_face(faces, clip, n_verts, f, radius, w, h, &fc, &bx0, &by0, &bw)
                        : 0u;
    const bool big = n_box > kDistLaneBox;
    const uint32_t n_px = big ? 0u : n_box;
    const uint32_t origin = n_px ? (uint32_t)by0 * w + (uint32_t)bx0 : 0u;
    for (uint32_t k = blockIdx.z; k < peels; k += gridDim.z) {
        const size_t layer = (size_t)blockIdx.y * peels + k;
        const float4 *rl = rs + layer * npx, *gl = gy + layer * npx;
        float acc[3][3] = {};  // corner, component (x, y, w)
        uint32_t n_hits = 0;
        BoxWalk at((uint32_t)bx0, (uint32_t)by0, bw, w, 0, 1);
        for (uint32_t p0 = 0; __any(p0 < n_px); p0 += kDistPx) {
            if (p0 < n_px) {
                uint32_t o[kDistPx];
                float2 yw[kDistPx];
#pragma unroll
                for (uint32_t s = 0; s < kDistPx; s++) {
                    const bool in = p0 + s < n_px;
                    o[s] = in ? at.o : origin;
                    at.next();
                    const float4 v = rl[o[s]];
                    yw[s] = make_float2(v.y, in ? v.w : 0.f);
                }
#pragma unroll
                for (uint32_t s = 0; s < kDistPx; s++) {
                    if (!(yw[s].y < 0.5f) && (uint32_t)(int64_t)(yw[s].x + 0.5f) == f) {
                        lds.hit_px[n_hits * 64 + lane] = o[s];
                        n_hits++;
                    }
                }
            }
            if (__any(p0 + kDistPx < n_px) && !__any(n_hits + kDistPx > kDistLaneHits)) {
                continue;
            }
            // (a lane reads what it wrote itself)
            for (uint32_t q = 0; __any(q < n_hits); q++) {
                const uint32_t px_o = q < n_hits ? lds.hit_px[q * 64 + lane] : 0u;
                const float g = q < n_hits ? gl[px_o].x : 0.f;
                if (g != 0.f) {
                    const uint32_t y = px_o / w, x = px_o - y * w;
                    const float px = (float)x + 0.5f, py = (float)y + 0.5f;
                    const TriDistE td = signed_dist_edge(px, py, fc.sx, fc.sy);
                    float4 t[3] = {};
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        add_corner(fc, td, px, py, c, g, W, H, &t[c]);
                    }
#pragma unroll
                    for (int r = 0; r < 3; r++) {
#pragma unroll
                        for (int c = 0; c < 3; c++) {
                            // a corner's row takes every corner of its vertex; a
                            // contribution left out is +0, as above
                            const bool add = c == r || fc.idx[c] == fc.idx[r];
                            acc[r][0] += add ? t[c].x : 0.f;
                            acc[r][1] += add ? t[c].y : 0.f;
                            acc[r][2] += add ? t[c].w : 0.f;
                        }
                    }
                }
            }
            n_hits = 0;
        }
        const uint64_t all = __ballot(big);
        if (all) {
            uint32_t at = 0;
            if (lane == 0) {
                at = atomicAdd(bigs.n, (uint32_t)__popcll(all));
            }
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) +
                 (uint32_t)__popcll(all & ((1ull << lane) - 1ull));
            if (big) {
                bigs.list[at] = make_uint2(f, (uint32_t)layer);
            }
        }
        if (f >= n_faces || big) {
            continue;
        }
        if (!ROWS) {
#pragma unroll
            for (int q = 0; q < 9; q++) {
                g_corner[(layer * n_faces + f) * 9 + q] = acc[q / 3][q % 3];
            }
        } else if (n_box) {
#pragma unroll
            for (int r = 0; r < 3; r++) {
                uint32_t d = 0;
                for (; d < max_deg; d++) {
                    const float fv = vf[(size_t)d * n_verts + fc.idx[r]];
                    if (fv >= -0.5f && (uint32_t)(int64_t)(fv + 0.5f) == f) {
                        break;
                    }
                }
                if (d < max_deg) {
                    float* dst = (float*)&out[(size_t)d * n_verts + fc.idx[r]];
                    dst[0] = acc[r][0];
                    dst[1] = acc[r][1];
                    dst[3] = acc[r][2];
                }
            }
        }
    }
}

// ColSum of the vertex's rows per peel, the peels' contributions (the last
// peel first), the z remap's transpose (the gradient's z is 0). One thread
// per vertex and component.
__global__ __launch_bounds__(256) void k_surface_soft_bwd_vtx(
        const float* g_corner, uint32_t peels, const float* faces, uint32_t n_faces,
        const float* vf, uint32_t n_verts, uint32_t max_deg, float* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_verts * 4) {
        return;
    }
    const uint32_t v = i >> 2, comp = i & 3u;
    float* dst = out + (size_t)blockIdx.y * n_verts * 4 + i;
    if (comp == 2) {
        *dst = 0.f;
        return;
    }
    const uint32_t c = comp == 3 ? 2u : comp;
    ContribSum total;
    for (uint32_t k = peels; k-- > 0;) {
        const float* g = g_corner + ((size_t)blockIdx.y * peels + k) * n_faces * 9;
        float acc = 0.f;
        for (uint32_t d = 0; d < max_deg; d++) {
            const float fv = vf[(size_t)d * n_verts + v];
            const uint32_t f = fv < -0.5f ? n_faces : fid_u(fv);
            if (f >= n_faces) {
                continue;
            }
            uint32_t q = 2;
            q = fid_u(faces[(size_t)f * 3 + 1]) == v ? 1u : q;
            q = fid_u(faces[(size_t)f * 3 + 0]) == v ? 0u : q;
            acc += g[(size_t)f * 9 + q * 3 + c];
        }
        total.push(acc);
    }
    *dst = total.sum();
}

// {V,1} layout, one thread per vertex: the union of its incident faces'
// soft bboxes in raster order, pixels whose face is incident to it.
__global__ __launch_bounds__(128) void k_gather_dist_grad_vtx(
        const float4* gy, const float4* rs, const float4* clip, uint32_t n_verts,
        const float* faces, uint32_t n_faces, const float* vf, uint32_t max_deg, float radius,
        uint32_t w, uint32_t h, uint32_t* err, float4* out) {
    const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= n_verts) {
        return;
    }
    const float W = (float)w, H = (float)h;
    int ux0 = (int)w, uy0 = (int)h, ux1 = -1, uy1 = -1;
    for (uint32_t d = 0; d < max_deg; d++) {
        const float fv = vf[(size_t)d * n_verts + u];
        if (fv < -0.5f) {
            continue;
        }
        const uint32_t f = (uint32_t)(int64_t)(fv + 0.5f);
        FaceCorners fc;
        int bx0, by0, bx1, by1;
        if (f >= n_faces) {
            atomicOr(err, 2u);
        } else if (load_face(faces, clip, n_verts, f, W, H, &fc, err) &&
                   soft_bbox(fc, w, h, radius, &bx0, &by0, &bx1, &by1)) {
            ux0 = min(ux0, bx0);
            uy0 = min(uy0, by0);
            ux1 = max(ux1, bx1);
            uy1 = max(uy1, by1);
        }
    }
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int y = uy0; y <= uy1; y++) {
        for (int x = ux0; x <= ux1; x++) {
            const size_t o = (size_t)y * w + x;
            const float4 r = rs[o];
            if (r.w < 0.5f) {
                continue;
            }
            const float g = gy[o].x;
            if (g == 0.f) {
                continue;
            }
            const uint32_t f = (uint32_t)(int64_t)(r.y + 0.5f);
            bool inc = false;
            for (uint32_t d = 0; d < max_deg && !inc; d++) {
                const float fv = vf[(size_t)d * n_verts + u];
                inc = fv >= -0.5f && (uint32_t)(int64_t)(fv + 0.5f) == f;
            }
            FaceCorners fc;
            if (!inc || f >= n_faces || !load_face(faces, clip, n_verts, f, W, H, &fc, err)) {
                continue;
            }
            const float px = (float)x + 0.5f, py = (float)y + 0.5f;
            const TriDistE td = signed_dist_edge(px, py, fc.sx, fc.sy);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if (fc.idx[k] == u) {
                    add_corner(fc, td, px, py, k, g, W, H, &acc);
                }
            }
        }
    }
    out[u] = acc;
}

}  // namespace
}  // namespace dressi

using namespace dressi;

// Whether `n` faces (times items and peels) of a mesh go by lanes. A wave for
// every face starts at about 1 ns, and that is what many small ones take: two
// 256 x 256 views of 327 680 faces 792 us, the thread per row before the waves
// 459, lanes 145; eight 64 x 64 ones of 20 480 219, 503 and 69. Where the boxes
// are large the lanes' pass is in vain (one 2048 x 2048 view of 327 680 faces
// 567 -> 678 us; the thread per row 5435), but their size is not known here (a
// sixteenth of that screen 435 -> 211): below 131 072 lanes are taken where
// the mesh has more faces than the screen has pixels.
static bool dist_by_lane(uint64_t n, uint32_t n_faces, uint32_t w, uint32_t h) {
    return n < (1ull << 32) &&
           (n >= 131072 || (n >= 16384 && (uint64_t)w * h < n_faces));
}
// Waves of k_dist_big (8192 of them take 762 us for the 678 above).
constexpr uint32_t kDistBigWaves = 32768;
constexpr int kDistBigSlot = 14;

template <bool ROWS>
static int launch_dist_lanes(dressi_ctx* ctx, const float* gy, const float* rs, uint32_t peels,
                             const float* clip, uint32_t n_verts, uint32_t n_items,
                             const float* faces, uint32_t n_faces, const float* vf,
                             uint32_t max_deg, float radius, uint32_t w, uint32_t h,
                             float* g_corner, float* out) {
    const uint64_t n = (uint64_t)n_faces * n_items * peels;
    void* ws = nullptr;
    if (int rc = ctx_workspace(ctx, kDistBigSlot, 8 + sizeof(uint2) * n, &ws)) return rc;
    const DistBig bigs{(uint32_t*)ws, (uint2*)((char*)ws + 8)};
    if (int rc = launch_zero(ctx->stream, ws, 8)) return rc;
    hipLaunchKernelGGL(k_dist_lanes<ROWS>,
                       dim3(div_up(n_faces, 64), n_items, std::min(peels, 16u)), dim3(64), 0,
                       ctx->stream, (const float4*)gy, (const float4*)rs, peels,
                       (const float4*)clip, n_verts, faces, n_faces, vf, max_deg, radius, w, h,
                       bigs, g_corner, (float4*)out);
    DRESSI_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_dist_big<ROWS>, dim3((uint32_t)std::min<uint64_t>(n, kDistBigWaves)), dim3(64), 0,
                       ctx->stream, (const float4*)gy, (const float4*)rs, peels,
                       (const float4*)clip, n_verts, faces, n_faces, vf, max_deg, radius, w, h,
                       bigs, g_corner, (float4*)out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

extern "C" int dressi_gather_dist_grad(dressi_ctx* ctx, const float* gy, const float* rs,
                                       const float* clip, uint32_t n_verts, const float* faces,
                                       uint32_t n_faces, const float* vtx_faces, uint32_t max_deg,
                                       float radius_px, int wide, uint32_t width, uint32_t height,
                                       float* out) {
    DRESSI_REQUIRE(ctx && gy && rs && clip && faces && vtx_faces && out, "bad arguments");
    DRESSI_REQUIRE(radius_px > 0.f, "radius_px must be > 0");
    DRESSI_REQUIRE(max_deg >= 1, "max_deg must be >= 1");
    DRESSI_REQUIRE((uint64_t)max_deg * n_verts < (1ull << 31), "adjacency too large");
    DRESSI_REQUIRE(!wide || (uint64_t)width * height <= kMaxImagePixels, "screen too large");
    if (!n_verts) return DRESSI_OK;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    if (wide) {
        hipLaunchKernelGGL(k_gather_dist_grad_rows, dim3(div_up(max_deg * n_verts, 256)),
                           dim3(256), 0, ctx->stream, faces, n_verts, n_faces, vtx_faces, max_deg,
                           ctx->d_err, (float4*)out);
        DRESSI_CHECK_LAUNCH();
        if (n_faces) {
            if (dist_by_lane(n_faces, n_faces, width, height)) {
                return launch_dist_lanes<true>(ctx, gy, rs, 1, clip, n_verts, 1, faces, n_faces,
                                               vtx_faces, max_deg, radius_px, width, height,
                                               nullptr, out);
            } else {
                hipLaunchKernelGGL(k_gather_dist_grad_faces, dim3(n_faces), dim3(64), 0,
                                   ctx->stream, (const float4*)gy, (const float4*)rs,
                                   (const float4*)clip, n_verts, faces, vtx_faces, max_deg,
                                   radius_px, width, height, (float4*)out);
            }
        }
    } else {
        hipLaunchKernelGGL(k_gather_dist_grad_vtx, dim3(div_up(n_verts, 128)), dim3(128), 0,
                           ctx->stream, (const float4*)gy, (const float4*)rs, (const float4*)clip,
                           n_verts, faces, n_faces, vtx_faces, max_deg, radius_px, width, height,
                           ctx->d_err, (float4*)out);
    }
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

extern "C" int dressi_surface_soft_bwd(dressi_ctx* ctx, const float* gy, const float* rs,
                                       uint32_t peels, const float* pos, uint32_t n_verts,
                                       uint32_t n_items, const float* faces, uint32_t n_faces,
                                       const float* vtx_faces, uint32_t n_rows, uint32_t max_deg,
                                       float radius_px, uint32_t width, uint32_t height,
                                       float* g_corner, float* out) {
    DRESSI_REQUIRE(ctx && gy && rs && pos && (faces || n_faces == 0) && vtx_faces && out &&
                           (g_corner || n_faces == 0),
                   "rasterize_soft backward: NULL buffer");
    DRESSI_REQUIRE(radius_px > 0.f, "radius_px must be > 0");
    DRESSI_REQUIRE(peels >= 1 && n_items <= kMaxBatchItems, "batch of %u items exceeds %u",
                   n_items, kMaxBatchItems);
    DRESSI_REQUIRE((uint64_t)width * height <= kMaxImagePixels && n_rows < (1u << 30),
                   "rasterize_soft backward: too large");
    if (!n_items || !n_rows) return DRESSI_OK;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    if (n_faces) {
        const uint32_t z = std::min(peels, 16u);
        if (dist_by_lane((uint64_t)n_faces * n_items * peels, n_faces, width, height)) {
            if (int rc = launch_dist_lanes<false>(ctx, gy, rs, peels, pos, n_verts, n_items, faces,
                                                  n_faces, nullptr, 0, radius_px, width, height,
                                                  g_corner, nullptr)) return rc;
        } else {
            hipLaunchKernelGGL(k_surface_soft_bwd_faces, dim3(n_faces, n_items, z), dim3(64), 0,
                               ctx->stream, (const float4*)gy, (const float4*)rs, peels,
                               (const float4*)pos, n_verts, faces, n_faces, radius_px, width,
                               height, g_corner);
        }
        DRESSI_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_surface_soft_bwd_vtx, dim3(div_up(n_rows * 4, 256), n_items), dim3(256),
                       0, ctx->stream, (const float*)g_corner, peels, faces, n_faces, vtx_faces,
                       n_rows, max_deg, out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}
