// surface.hip -- the torch surface's ops (opendressi_amd/torch) as kernels
// of their own: each does in a few launches (one for most, up to six for the
// texture gradient) what the surface composed from the per-op entry points and
// torch's elementwise kernels, with the same float operations in the same
// order (python/dressi/torch/ops.py:95-698 and the reference's backward
// kernels it runs). Images are [item][H][W][C], `rast` is the surface's
// raster, VEC4 (u, v, z / w, face + 1); face lists are float ids {F,3},
// adjacencies {max_deg, V} (VertexFacesTex) of the same faces.
//
// A call of the surface used to be 10-20 launches of a few microseconds each
// (a slice, a product, a copy), bound by the host that issued them and by
// reading and writing each intermediate image.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "internal.h"
#include "surface_core.h"

namespace dressi {
namespace {

// ---------------------------------------------------------------------------
// interpolate
// ---------------------------------------------------------------------------

// out = u a0 + v a1 + ((1 - u) - v) a2 of the pixel's face corners
// (LookupFaces + FaceFetch per corner; 0 for a pixel without a face), one
// thread per pixel. Bound by the raster's 16 bytes and the C values out.
template <int C>
__global__ __launch_bounds__(256) void k_surface_interp(const float* attr, size_t attr_stride,
                                                        uint32_t n_attr, const float4* rast,
                                                        size_t npx, const float* faces,
                                                        uint32_t n_faces, uint32_t* err,
                                                        float* out) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npx) {
        return;
    }
    attr += blockIdx.y * attr_stride;
    rast += blockIdx.y * npx;
    out += blockIdx.y * npx * C;
    const float4 r = rast[p];
    const int f = (int)(r.w + 0.5f) - 1;
    float a[3][C];
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int c = 0; c < C; c++) {
            a[k][c] = 0.f;
        }
    }
    if (f >= 0 && (uint32_t)f < n_faces) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const uint32_t vi = fid_u(faces[(size_t)f * 3 + k]);
            if (vi >= n_attr) {
                atomicOr(err, 32u);
                continue;
            }
#pragma unroll
            for (int c = 0; c < C; c++) {
                a[k][c] = attr[(size_t)vi * C + c];
            }
        }
    }
    const float w2 = (1.f - r.x) - r.y;
#pragma unroll
    for (int c = 0; c < C; c++) {
        out[p * C + c] = r.x * a[0][c] + r.y * a[1][c] + w2 * a[2][c];
    }
}

// FaceFetchBwd (f_ops.cpp:1631-1733, n = 0: every pixel of the face's box
// that shows it, in raster order) of g u, g v and g ((1 - u) - v), the three
// corners' gradients together: g_face {N,F,3} VEC C.
//
// G lanes per face and item: PX G pixels of the box at once, the few that show
// the face form their terms side by side, and one lane per corner and
// channel adds them in order. One thread per face walked its box pixel by
// pixel at a load latency each, three times over (one call per corner):
// 3 x 515 us for four 1280 x 720 views of 20 480 faces, where a wave per face
// takes 70. More pixels per step cost the LDS that keeps waves resident (four
// per lane: 107 us there).
//
// Screen pixels per face from which a face gets a wave of its own. Below, its
// box is a few steps of 32 pixels and four faces share a wave. Sixteen lanes
// and a wave per face take (both kernels of the gradient) 41 and 62 us for
// four 256 x 256 views at 3 pixels per face, 36 and 37 at 13, 49 and 35 at
// 51; for four 1280 x 720 views 90 and 93 at 45, 459 and 163 at 720.
constexpr uint32_t kInterpWavePx = 32;

template <int C, int G>
__global__ __launch_bounds__(64) void k_surface_interp_bwd_faces(
        const float* gy, const float4* rast, uint32_t w, uint32_t h, const float4* clip,
        size_t clip_stride, const float* faces, uint32_t n_faces, uint32_t n_verts,
        float* g_face) {
    static_assert(3 * C <= G, "a lane per corner and channel");
    constexpr uint32_t PX = 2;  // pixels per lane and step
    __shared__ float term[64 / G][G * PX][3 * C];
    const uint32_t lane = threadIdx.x % G, grp = threadIdx.x / G;
    const uint32_t f = blockIdx.x * (64 / G) + grp;
    const bool live = f < n_faces;
    const size_t npx = (size_t)w * h;
    gy += blockIdx.y * npx * C;
    rast += blockIdx.y * npx;
    clip += blockIdx.y * clip_stride;
    float s[3][2];
    bool ok = live;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const uint32_t v = live ? fid_u(faces[(size_t)f * 3 + k]) : n_verts;
        const float4 c = v < n_verts ? clip[v] : make_float4(0.f, 0.f, 0.f, 0.f);
        ok = ok && c.w > 1e-6f;
        s[k][0] = (c.x / c.w * 0.5f + 0.5f) * (float)w;
        s[k][1] = (c.y / c.w * 0.5f + 0.5f) * (float)h;
    }
    int x0 = (int)floorf(smin(smin(s[0][0], s[1][0]), s[2][0]) - 1.f);
    int x1 = (int)ceilf(smax(smax(s[0][0], s[1][0]), s[2][0]) + 1.f);
    int y0 = (int)floorf(smin(smin(s[0][1], s[1][1]), s[2][1]) - 1.f);
    int y1 = (int)ceilf(smax(smax(s[0][1], s[1][1]), s[2][1]) + 1.f);
    x0 = x0 > 0 ? x0 : 0;
    y0 = y0 > 0 ? y0 : 0;
    x1 = x1 < (int)w - 1 ? x1 : (int)w - 1;
    y1 = y1 < (int)h - 1 ? y1 : (int)h - 1;
    ok = ok && x1 >= x0 && y1 >= y0;
    const uint32_t bw = ok ? (uint32_t)(x1 - x0 + 1) : 1u;
    const uint32_t n_px = ok ? bw * (uint32_t)(y1 - y0 + 1) : 0u;
    const uint32_t origin = ok ? (uint32_t)y0 * w + (uint32_t)x0 : 0u;
    BoxWalk at(ok ? (uint32_t)x0 : 0u, ok ? (uint32_t)y0 : 0u, bw, w, lane, G);
    const uint64_t below = (1ull << lane) - 1ull;
    float acc = 0.f;
    for (uint32_t p0 = 0; __any(p0 < n_px); p0 += G * PX) {
        float4 r[PX];
        uint32_t o[PX];
#pragma unroll
        for (uint32_t q = 0; q < PX; q++) {
            const bool in = p0 + q * G + lane < n_px;
            o[q] = in ? at.o : origin;
            at.next();
            r[q] = rast[o[q]];
            r[q].w = in ? r[q].w : 0.f;
        }
        uint32_t n_hits = 0;
#pragma unroll
        for (uint32_t q = 0; q < PX; q++) {
            const bool hit = live && fid_u(r[q].w) == f + 1;
            // the group's lanes of the ballot
            const uint64_t m = (__ballot(hit) >> (grp * G)) & (~0ull >> (64 - G));
            if (hit) {
                const uint32_t slot = n_hits + (uint32_t)__popcll(m & below);
                const float w2 = (1.f - r[q].x) - r[q].y;
#pragma unroll
                for (int c = 0; c < C; c++) {
                    const float g = gy[(size_t)o[q] * C + c];
                    term[grp][slot][c] = g * r[q].x;
                    term[grp][slot][C + c] = g * r[q].y;
                    term[grp][slot][2 * C + c] = g * w2;
                }
            }
            n_hits += (uint32_t)__popcll(m);
        }
        wave_lds_fence();
        if (lane < 3 * C) {
#pragma unroll 16
            for (uint32_t q = 0; q < n_hits; q++) {
                acc += term[grp][q][lane];
            }
        }
        wave_lds_fence();
    }
    if (live && lane < 3 * C) {
        g_face[((size_t)blockIdx.y * n_faces + f) * 3 * C + lane] = acc;
    }
}

// LookupFacesBwd (f_ops.cpp:1521-1565) of each corner and the sum of the
// contributions: per item corners 2, 1, 0 (newest first); one attribute
// shared by the items takes every item's, the last item first. One thread
// per vertex and channel (and item, where the attribute is per item).
template <int C>
__global__ __launch_bounds__(256) void k_surface_interp_bwd_vtx(
        const float* g_face, const float* faces, uint32_t n_faces, const float* vf,
        uint32_t n_verts, uint32_t max_deg, uint32_t n_items, int shared_attr, float* g_attr) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_verts * C) {
        return;
    }
    const uint32_t v = i / C, c = i - v * C;
    const size_t item_stride = (size_t)n_faces * 3 * C;
    constexpr int kItems = 4;  // items walked together: one look at the adjacency
    ContribSum total;
    const uint32_t first = shared_attr ? 0u : blockIdx.y;
    const uint32_t last = shared_attr ? n_items : blockIdx.y + 1;
    for (uint32_t hi = last; hi > first;) {
        const uint32_t n = hi - first < (uint32_t)kItems ? hi - first : (uint32_t)kItems;
        float acc[kItems][3] = {};
        for (uint32_t d = 0; d < max_deg; d++) {
            const float fv = vf[(size_t)d * n_verts + v];
            if (fv < -0.5f) {
                continue;
            }
            const uint32_t f = fid_u(fv);
            if (f >= n_faces) {
                continue;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if (fid_u(faces[(size_t)f * 3 + k]) == v) {
#pragma unroll
                    for (int t = 0; t < kItems; t++) {
                        if ((uint32_t)t < n) {
                            acc[t][k] += g_face[(size_t)(hi - 1 - t) * item_stride +
                                                ((size_t)f * 3 + k) * C + c];
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kItems; t++) {
            if ((uint32_t)t < n) {
                total.push(acc[t][2]);
                total.push(acc[t][1]);
                total.push(acc[t][0]);
            }
        }
        hi -= n;
    }
    g_attr[(size_t)first * n_verts * C + i] = total.sum();
}

int check_surface(dressi_ctx* ctx, uint32_t n_comp, uint32_t w, uint32_t h, uint32_t n_items) {
    DRESSI_REQUIRE(ctx != nullptr, "NULL context");
    DRESSI_REQUIRE(n_comp >= 1 && n_comp <= 4, "n_comp must be 1..4");
    DRESSI_REQUIRE((uint64_t)w * h <= kMaxImagePixels, "screen too large");
    DRESSI_REQUIRE(n_items <= kMaxBatchItems, "batch of %u items exceeds %u", n_items,
                   kMaxBatchItems);
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    return DRESSI_OK;
}

// Calls `fn` with the channel count as a constant.
template <typename Fn>
void with_channels(uint32_t n_comp, Fn&& fn) {
    switch (n_comp) {
        case 1: fn(std::integral_constant<int, 1>{}); break;
        case 2: fn(std::integral_constant<int, 2>{}); break;
        case 3: fn(std::integral_constant<int, 3>{}); break;
        default: fn(std::integral_constant<int, 4>{}); break;
    }
}

}  // namespace
}  // namespace dressi

using namespace dressi;

extern "C" {

int dressi_surface_interpolate(dressi_ctx* ctx, const float* attr, uint32_t n_attr,
                               uint32_t n_comp, int attr_per_item, const float* rast,
                               uint32_t width, uint32_t height, uint32_t n_items,
                               const float* faces, uint32_t n_faces, float* out) {
    if (int rc = check_surface(ctx, n_comp, width, height, n_items)) return rc;
    DRESSI_REQUIRE((attr || n_attr == 0) && rast && (faces || n_faces == 0) && out,
                   "interpolate: NULL buffer");
    const size_t npx = (size_t)width * height;
    if (!npx || !n_items) return DRESSI_OK;
    with_channels(n_comp, [&](auto c) {
        hipLaunchKernelGGL(k_surface_interp<decltype(c)::value>,
                           dim3((uint32_t)((npx + 255) / 256), n_items), dim3(256), 0, ctx->stream,
                           attr, attr_per_item ? (size_t)n_attr * n_comp : (size_t)0, n_attr,
                           (const float4*)rast, npx, faces, n_faces, ctx->d_err, out);
    });
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_surface_interpolate_bwd(dressi_ctx* ctx, const float* gy, uint32_t n_comp,
                                   const float* rast, uint32_t width, uint32_t height,
                                   uint32_t n_items, const float* clip, uint32_t n_clip,
                                   int clip_per_item, const float* faces, uint32_t n_faces,
                                   const float* vtx_faces, uint32_t n_verts, uint32_t max_deg,
                                   int shared_attr, float* g_face, float* g_attr) {
    if (int rc = check_surface(ctx, n_comp, width, height, n_items)) return rc;
    DRESSI_REQUIRE(gy && rast && (clip || n_clip == 0) && (faces || n_faces == 0) &&
                           (vtx_faces || n_verts == 0) && (g_face || n_faces == 0) && g_attr,
                   "interpolate backward: NULL buffer");
    DRESSI_REQUIRE((uint64_t)n_verts * n_comp < (1ull << 32), "too many vertices");
    if (!n_items || !n_verts) return DRESSI_OK;
    with_channels(n_comp, [&](auto c) {
        constexpr int C = decltype(c)::value;
        if (n_faces) {
            const auto launch = [&](auto kernel, uint32_t per_wave) {
                hipLaunchKernelGGL(kernel, dim3(div_up(n_faces, per_wave), n_items), dim3(64), 0,
                                   ctx->stream, gy, (const float4*)rast, width, height,
                                   (const float4*)clip, clip_per_item ? (size_t)n_clip : (size_t)0,
                                   faces, n_faces, n_clip, g_face);
            };
            if ((uint64_t)width * height < (uint64_t)n_faces * kInterpWavePx) {
                launch(k_surface_interp_bwd_faces<C, 16>, 4);
            } else {
                launch(k_surface_interp_bwd_faces<C, 64>, 1);
            }
        }
        hipLaunchKernelGGL(k_surface_interp_bwd_vtx<C>,
                           dim3(div_up(n_verts * n_comp, 256), shared_attr ? 1 : n_items),
                           dim3(256), 0, ctx->stream, g_face, faces, n_faces, vtx_faces, n_verts,
                           max_deg, n_items, shared_attr, g_attr);
    });
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

}  // extern "C"
