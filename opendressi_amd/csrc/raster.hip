// raster.hip -- tile binning, the per-op rasterizers (RasterizeSoft,
// Rasterize, RasterizeFaceId) and SoftClip.
#include <algorithm>
#include <mutex>

#include "raster_core.h"
#include "soft_clip.h"

namespace dressi {

// ---------------------------------------------------------------------------
// Binning
// ---------------------------------------------------------------------------

// A hard bin's list holds kHardBinShare times the faces that a bin would have
// if every view's were spread evenly over its tiles, and kHardBinMin more: a
// closed mesh that fills a third of the screen has about four times that
// share on a tile and up to eleven at its limb. Small problems get what
// kHardListEntries (16 MB) have room for, so that none of their lists fills up.
// The overflow takes kHardOverShare entries per face and view. Four 1280 x 720
// views of 20 480 faces take 23 MB, 64 of 1024 x 1024 and 81 920 faces 437 MB
// (their records 6.6 and 419).
constexpr uint64_t kHardBinShare = 8, kHardBinMin = 32, kHardOverShare = 4;
constexpr uint64_t kHardListEntries = 4ull << 20;
// Bins from which a list's least is 16 entries, and words for the chains' heads
// up to there (64 MB; a bin has at least eight): many bins are many pixels, of
// which few have full lists.
constexpr uint64_t kHardManyBins = 1ull << 20, kHardHeads = 1ull << 24;
// Neither grows past these (4 GB each); a list keeps at least 16 entries.
constexpr uint64_t kHardListMax = 1ull << 30, kHardOverMax = 1ull << 29;

HardBinSizes hard_bin_sizes(const RasterGeom& g) {
    const uint64_t n_bins = (uint64_t)g.n_tiles * g.n_views;
    const uint64_t faces = std::max<uint64_t>(g.n_faces, 1);
    uint64_t cap = std::max((n_bins > kHardManyBins ? 16 : kHardBinMin) +
                                    kHardBinShare * faces / g.n_tiles,
                            kHardListEntries / n_bins);
    cap = std::min(cap, std::max<uint64_t>(kHardListMax / n_bins, 16));
    cap = std::min(cap, faces);
    HardBinSizes z;
    z.n_bins = (uint32_t)n_bins;
    z.cap = (uint32_t)cap;
    z.over_cap = cap == faces ? 0u
                              : (uint32_t)std::min(faces * g.n_views * kHardOverShare + 4096,
                                                   kHardOverMax);
    z.chains = kHardChains;
    while (z.chains > 8 && n_bins * z.chains > kHardHeads) z.chains /= 2;
    z.bytes = sizeof(uint32_t) * (n_bins + 4 + 2 * (size_t)z.over_cap +
                                  n_bins * (cap + (z.over_cap ? z.chains : 0u)));
    return z;
}

void hard_bin_carve(void* base, const HardBinSizes& z, HardBinBuffers* b) {
    uint32_t* p = (uint32_t*)base;
    b->counts = p;
    b->n_over = p + z.n_bins;
    b->spilt = b->n_over + 1;
    p += ((size_t)z.n_bins + 3) & ~(size_t)1;  // pairs: 8-byte aligned
    b->over = (uint2*)p;
    p += 2 * (size_t)z.over_cap;
    b->heads = p;
    p += z.over_cap ? (size_t)z.n_bins * z.chains : 0;
    b->list = p;
    b->cap = z.cap;
    b->over_cap = z.over_cap;
    b->n_bins = z.n_bins;
    b->chains = z.chains;
}

// ---------------------------------------------------------------------------
// Hard rasterizer (Rasterize / RasterizeFaceId)
// ---------------------------------------------------------------------------

// Setup and binning, a thread per (view, face), from the reference's float
// face ids (decoded as RasterizeCore does, uint32_t(int64_t(x)); a bad one is
// reported) or from int32 ones. `gl`: clip z in [-w, w], remapped to
// 0.5 (z + w). b's counters are zero.
//
// Lists of a fixed size take a face where it is set up. With lists sized by a
// count and a scan (the form before) a raster had two launches more: 17 + 15
// + 18 us for four 1280 x 720 views of 20 480 faces, now 21. What bounds is
// the adds' round trip to memory: a wave shares its faces' tiles out evenly,
// a lane has kBinPairs of them on their way at once (a thread that goes
// through its own face's tiles, four at a time: 50 us). The lists' size makes
// no difference there (128 entries or the whole mesh).
//
// What finds its list full goes to chains of its own bin, which its tile then
// reads side by side, so that the work stays linear in the views (one overflow
// for all tiles, as it was before, took 33 ms for 64 1024 x 1024 views of
// 81 920 faces, which now take 2.3, and 169 ms for 128 of 512 x 512, now 4.3;
// counted, scanned and filled lists 4.1 and 6.7). Where nearly everything
// overflows, a mesh on nine tiles of each of 64 512 x 512 views: 7.6 ms, the
// scanned lists 9.7.
constexpr uint32_t kBinPairs = 4;

__global__ __launch_bounds__(256) void k_hard_setup_bin(RasterGeom g, const float4* clip,
                                                        uint32_t n_verts, const float* faces,
                                                        const int32_t* faces_i, int gl,
                                                        HardBinBuffers b, uint32_t* err,
                                                        HardRec* recs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < g.n_views * g.n_faces;
    const uint32_t view = live ? i / g.n_faces : 0u;
    const uint32_t f = live ? i - view * g.n_faces : 0u;
    HardRec r;
    r.bx0 = 1;
    r.bx1 = 0;
    r.by0 = 1;
    r.by1 = 0;
    if (live) {
        int idx[3];
        float4 c[3];
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const uint32_t v = faces ? (uint32_t)(int64_t)faces[(size_t)f * 3 + k]
                                     : (uint32_t)faces_i[(size_t)f * 3 + k];
            ok = ok && v < n_verts;
            idx[k] = (int)v;
        }
        if (ok) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                c[k] = clip[(size_t)view * n_verts + idx[k]];
                if (gl) {
                    c[k].z = 0.5f * (c[k].z + c[k].w);
                }
            }
            hard_setup(c, idx, g.width, g.height, &r);
        } else if (err) {
            atomicOr(err, 16u);
        }
        recs[i] = r;
    }
    const bool any = r.bx0 <= r.bx1 && r.by0 <= r.by1;
    const uint32_t tx0 = any ? (uint32_t)r.bx0 / kTile : 0u;
    const uint32_t ty0 = any ? (uint32_t)r.by0 / kTile : 0u;
    const uint32_t tw = any ? (uint32_t)r.bx1 / kTile - tx0 + 1 : 1u;
    const uint32_t n = any ? tw * ((uint32_t)r.by1 / kTile - ty0 + 1) : 0u;
    const uint32_t first = view * g.n_tiles + ty0 * g.tiles_x + tx0;
    // the wave's (face, tile) pairs, lane l's behind those of the lanes below
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t incl = n;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint32_t v = (uint32_t)__shfl_up((int)incl, o);
        incl += lane >= o ? v : 0u;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    for (uint32_t t0 = 0; t0 < total; t0 += 64 * kBinPairs) {
        uint32_t bin[kBinPairs], face[kBinPairs], slot[kBinPairs];
#pragma unroll
        for (uint32_t k = 0; k < kBinPairs; k++) {
            const uint32_t t = t0 + k * 64 + lane;
            uint32_t of = 0;  // the lanes whose pairs are all before t
#pragma unroll
            for (uint32_t step = 32; step >= 1; step >>= 1) {
                of += (uint32_t)__shfl((int)incl, (int)(of + step - 1)) <= t ? step : 0u;
            }
            const uint32_t at = t - (uint32_t)__shfl((int)(incl - n), (int)of);
            const uint32_t tw_of = (uint32_t)__shfl((int)tw, (int)of);
            face[k] = (uint32_t)__shfl((int)f, (int)of);
            const uint32_t ty = at / tw_of;
            bin[k] = (uint32_t)__shfl((int)first, (int)of) + ty * g.tiles_x + (at - ty * tw_of);
            slot[k] = t < total ? atomicAdd(&b.counts[bin[k]], 1u) : 0u;
        }
        uint64_t full[kBinPairs];  // the lanes whose bin's list is full
        uint32_t n_full = 0;
#pragma unroll
        for (uint32_t k = 0; k < kBinPairs; k++) {
            const bool in = t0 + k * 64 + lane < total;
            if (in && slot[k] < b.cap) {
                b.list[(size_t)bin[k] * b.cap + slot[k]] = face[k];
            }
            full[k] = __ballot(in && slot[k] >= b.cap);
            n_full += (uint32_t)__popcll(full[k]);
        }
        if (n_full) {
            // Places in the overflow, one add for the wave's; then each into
            // chain (slot - cap) % chains of its bin. A chain's length
            // follows from the bin's count, so heads need no initial value.
            uint32_t at = 0;
            if (lane == 0) {
                at = atomicAdd(b.n_over, n_full);
                if (at + n_full > b.over_cap) {
                    *b.spilt = 1u;
                }
            }
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll
            for (uint32_t k = 0; k < kBinPairs; k++) {
                const uint32_t o = at + (uint32_t)__popcll(full[k] & ((1ull << lane) - 1ull));
                if ((full[k] >> lane & 1u) && o < b.over_cap) {
                    const uint32_t chain = (slot[k] - b.cap) & (b.chains - 1);
                    b.over[o] = make_uint2(
                            face[k],
                            atomicExch(&b.heads[(size_t)bin[k] * b.chains + chain], o));
                }
                at += (uint32_t)__popcll(full[k]);
            }
        }
    }
}

int launch_hard_setup_bin(hipStream_t s, const RasterGeom& g, const float* clip, uint32_t n_verts,
                          const float* faces, const int32_t* faces_i, int gl,
                          const HardBinBuffers& b, uint32_t* err, HardRec* recs) {
    const uint32_t n = g.n_views * g.n_faces;
    if (n) {
        hipLaunchKernelGGL(k_hard_setup_bin, dim3(div_up(n, 256)), dim3(256), 0, s, g,
                           (const float4*)clip, n_verts, faces, faces_i, gl, b, err, recs);
        DRESSI_CHECK_LAUNCH();
    }
    return DRESSI_OK;
}

// One workgroup per (tile, view), a wave per 8x8 block of the tile. mode 0:
// perspective-correct attribute of the winner (cpu_raster.cpp:205-223), mode
// 1: face + 1, mode 2: (u, v, z / w, face + 1) of the torch surface's raster,
// whose `attr` are the clip positions {V} VEC4 (z, w read). n_attr > 1 (mode
// 0, one view): that many attribute sets of the one raster, `attr_view`
// floats apart, an image each.
//
// A wave folds only the records whose bbox meets its block, found by one
// test per lane and a ballot; with each wave walking all of the tile's
// records the raster of four 1280 x 720 views of 20 480 faces took 71 us,
// now 58: what is left is each tile's chain of dependent loads (a list's
// first entries are read beside its count).
// Records staged at once, 128 (10 KB): with 256 their LDS leaves seven
// workgroups to a CU instead of eight (61.5 us, now 56.5).
constexpr uint32_t kHardStage = 128;

__global__ __launch_bounds__(kTileThreads) void k_raster_hard(RasterGeom g, const HardRec* recs,
                                                              HardBinBuffers b,
                                                              const float* attr,
                                                              uint32_t n_comp, int mode,
                                                              float* out, size_t attr_view,
                                                              float* ids, uint32_t n_attr) {
    __shared__ HardRec lds_rec[kHardStage];
    __shared__ uint32_t lds_face[kHardStage];
    const uint32_t tile = blockIdx.x;
    const uint32_t view = blockIdx.y;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const int bx = (int)((tile % g.tiles_x) * kTile + (wave & 1u) * 8u);
    const int by = (int)((tile / g.tiles_x) * kTile + (wave >> 1) * 8u);
    const int px = bx + (int)(lane & 7u);
    const int py = by + (int)(lane >> 3);
    const HardRec* vrec = recs + (size_t)view * g.n_faces;
    uint64_t best = kEmptyKey;
    const uint32_t bin = view * g.n_tiles + tile;
    const uint32_t* list = b.list + (size_t)bin * b.cap;
    const uint32_t first =
            threadIdx.x < kHardStage && threadIdx.x < b.cap ? list[threadIdx.x] : 0u;
    const uint32_t n_bin = b.counts[bin];
    // a full list and a full overflow: every face of the view
    const bool full = n_bin > b.cap;
    const bool implicit = full && *b.spilt;
    const uint32_t n_list = implicit ? g.n_faces : full ? b.cap : n_bin;
    // folds the `cnt` staged records
    const auto fold = [&](uint32_t cnt) {
        for (uint32_t q = 0; q < cnt; q += 64) {
            const HardRec& mine = lds_rec[q + lane < cnt ? q + lane : q];
            uint64_t m = __ballot(q + lane < cnt && mine.bx0 <= bx + 7 && mine.bx1 >= bx &&
                                  mine.by0 <= by + 7 && mine.by1 >= by);
            for (; m; m &= m - 1) {
                const uint32_t j = q + (uint32_t)__builtin_ctzll(m);
                hard_fragment(lds_rec[j], lds_face[j], px, py, &best);
            }
        }
    };
    for (uint32_t base = 0; base < n_list; base += kHardStage) {
        const uint32_t cnt = (n_list - base) < kHardStage ? (n_list - base) : kHardStage;
        if (base) {
            __syncthreads();
        }
        if (threadIdx.x < cnt) {
            const uint32_t at = base + threadIdx.x;
            const uint32_t f = implicit ? at : base == 0 ? first : list[at];
            lds_face[threadIdx.x] = f;
            lds_rec[threadIdx.x] = vrec[f];
        }
        __syncthreads();
        fold(cnt);
    }
    if (full && !implicit) {
        // the bin's chains side by side: entry r of chain c is its overflow
        // face c + r chains, counted from the chain's head
        static_assert(kHardChains <= kHardStage, "a record staged per chain");
        const uint32_t n_over = n_bin - b.cap;
        uint32_t at = threadIdx.x < b.chains && threadIdx.x < n_over
                              ? b.heads[(size_t)bin * b.chains + threadIdx.x]
                              : 0u;
        for (uint32_t base = 0; base < n_over; base += b.chains) {
            const uint32_t cnt = (n_over - base) < b.chains ? (n_over - base) : b.chains;
            __syncthreads();
            if (threadIdx.x < cnt) {
                const uint2 e = b.over[at];
                at = e.y;
                lds_face[threadIdx.x] = e.x;
                lds_rec[threadIdx.x] = vrec[e.x];
            }
            __syncthreads();
            fold(cnt);
        }
    }
    if (px >= (int)g.width || py >= (int)g.height) {
        return;
    }
    const size_t o = ((size_t)view * g.height + py) * g.width + px;
    const float id = best == kEmptyKey ? 0.f : (float)key_face(best) + 1.f;
    if (ids) {
        ids[o] = id;
    }
    if (mode == 1) {
        out[o] = id;
        return;
    }
    const size_t out_attr = (size_t)g.width * g.height * n_comp;
    if (best == kEmptyKey) {
        for (uint32_t a = 0; a < n_attr; a++) {
            for (uint32_t c = 0; c < n_comp; c++) {
                out[a * out_attr + o * n_comp + c] = 0.f;
            }
        }
        return;
    }
    attr += (size_t)view * attr_view;
    const HardRec& r = vrec[key_face(best)];
    float l[3];
    barycentric((float)px + 0.5f, (float)py + 0.5f, r.x[0], r.y[0], r.x[1], r.y[1], r.x[2],
                r.y[2], r.inv_area, &l[0], &l[1], &l[2]);
    const float denom = l[0] * r.inv_w[0] + l[1] * r.inv_w[1] + l[2] * r.inv_w[2];
    if (mode == 2) {
        // attributes (1, 0), (0, 1), (0, 0), clip z and w by the same sums
        float num[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float4 c = ((const float4*)attr)[r.idx[k]];
            const float a[4] = {k == 0 ? 1.f : 0.f, k == 1 ? 1.f : 0.f, c.z, c.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                num[q] += l[k] * r.inv_w[k] * a[q];
            }
        }
        ((float4*)out)[o] = make_float4(num[0] / denom, num[1] / denom,
                                        (num[2] / denom) / (num[3] / denom), id);
        return;
    }
    for (uint32_t a = 0; a < n_attr; a++, attr += attr_view, out += out_attr) {
        for (uint32_t c = 0; c < n_comp; c++) {
            float num = 0.f;
            for (int k = 0; k < 3; k++) {
                num += l[k] * r.inv_w[k] * attr[(size_t)r.idx[k] * n_comp + c];
            }
            out[o * n_comp + c] = num / denom;
        }
    }
}

int launch_raster_hard(hipStream_t s, const RasterGeom& g, const HardRec* recs,
                       const HardBinBuffers& b, const float* attr, uint32_t n_comp, int mode,
                       float* out, size_t attr_view, float* ids, uint32_t n_attr) {
    hipLaunchKernelGGL(k_raster_hard, dim3(g.n_tiles, g.n_views), dim3(kTileThreads), 0, s, g,
                       recs, b, attr, n_comp, mode, out, attr_view, ids, n_attr);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

// ---------------------------------------------------------------------------
// Per-op soft rasterizer (RasterizeSoft)
// ---------------------------------------------------------------------------

// Fill kernel for counters (graph-capture safe, unlike a memset node).
__global__ void k_fill_u32(uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

// One thread per face: soft corners via faces_soft, face id from the last
// soft corner, hard corners via faces_tex[hard face] (cpu_raster.cpp:257-303);
// the face is appended to the fixed-capacity bins of the tiles its soft
// pixel bbox touches.
__global__ __launch_bounds__(256) void k_soft_setup_op(RasterGeom g, const float4* soft_clip,
                                                        const float* face_id,
                                                        const float* faces_soft,
                                                        const float4* hard_clip,
                                                        uint32_t n_verts,
                                                        const float* faces_tex, BinBuffers b,
                                                        uint32_t* err, SoftRec* recs,
                                                        CullRec* cull) {
    __shared__ BinLds blds;
    const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
    SoftRec r;
    r.bx0 = 1;
    r.bx1 = 0;
    r.by0 = 1;
    r.by1 = 0;
    r.flags = 0;
    if (f < g.n_faces) {
        float4 sc[3], hc[3];
        float fid = 0.f;
        bool ok = true;
        const uint32_t n_soft = 3 * g.n_faces;
        for (int k = 0; k < 3 && ok; k++) {
            const uint32_t vi = (uint32_t)(int64_t)faces_soft[(size_t)f * 3 + k];
            if (vi >= n_soft) {
                atomicOr(err, 1u);
                ok = false;
                break;
            }
            sc[k] = soft_clip[vi];
            if (!clip_w_valid(sc[k].w)) {
                ok = false;  // the reference skips the face at the first bad corner
                break;
            }
            fid = face_id[vi];
        }
        const uint32_t hf = ok ? fid_u(fid) : 0u;
        if (ok && hf >= g.n_faces) {
            atomicOr(err, 2u);
            ok = false;
        }
        for (int k = 0; k < 3 && ok; k++) {
            const uint32_t vi = fid_u(faces_tex[(size_t)hf * 3 + k]);
            if (vi >= n_verts) {
                atomicOr(err, 4u);
                ok = false;
                break;
            }
            hc[k] = hard_clip[vi];
        }
        if (ok) {
            soft_setup(sc, hc, fid, g.width, g.height, &r);
        }
        recs[f] = r;
        cull[f] = cull_setup(r);
    }
    const bool valid = f < g.n_faces && r.bx0 <= r.bx1 && r.by0 <= r.by1;
    bin_append(b, g, valid, 0u, f, r.bx0, r.by0, r.bx1, r.by1, soft_bin_tri(r), blds);
}

// One wave per 8x8 block: resolves the winner, then re-evaluates its signed
// distance and hard z (the output channels) from its record.
__global__ __launch_bounds__(64) void k_raster_soft_op(RasterGeom g, const SoftRec* recs,
                                                       const CullRec* cull, BinBuffers b,
                                                       float radius, const float* prev,
                                                       float4* out) {
    const BlockPos blk = block_pos(blockIdx.x, g);
    if (!blk.valid) {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int px = blk.bx + (lane & 7);
    const int py = blk.by + (lane >> 3);
    const BinView bv = bin_view(b, blk.tile, g.n_faces);
    __shared__ ResolveLds lds;
    const PixelBest best =
            resolve_block(recs, cull, bv, blk.bx, blk.by, radius, prev, g.width, lds);
    if (px >= (int)g.width || py >= (int)g.height) {
        return;
    }
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    if (best.key != kEmptyKey) {
        const SoftRec& r = recs[key_face(best.key)];
        const float p0 = (float)px + 0.5f;
        const float p1 = (float)py + 0.5f;
        const float dist = signed_dist(p0, p1, r.hx, r.hy, r.ex, r.ey, r.len2);
        o = make_float4(dist, r.fid, hard_z_at(r, p0, p1), 1.f);
    }
    out[(size_t)py * g.width + px] = o;
}

// The torch surface's soft raster: SoftClip and the soft setup of every item's
// faces from its clip positions (z in [-w, w], remapped), binned per item.
__global__ __launch_bounds__(256) void k_surface_soft_setup(RasterGeom g, const float4* pos,
                                                            uint32_t n_verts, const float* faces,
                                                            float radius, BinBuffers b,
                                                            uint32_t* err, SoftRec* recs,
                                                            CullRec* cull) {
    __shared__ BinLds blds;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < g.n_views * g.n_faces;
    const uint32_t view = live ? i / g.n_faces : 0;
    const uint32_t f = live ? i - view * g.n_faces : 0;
    SoftRec r;
    r.bx0 = 1;
    r.bx1 = 0;
    r.by0 = 1;
    r.by1 = 0;
    r.flags = 0;
    if (live) {
        float4 hc[3], sc[3];
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const uint32_t v = fid_u(faces[(size_t)f * 3 + k]);
            ok = ok && v < n_verts;
            hc[k] = ok ? pos[(size_t)view * n_verts + v] : make_float4(0.f, 0.f, 0.f, 0.f);
            hc[k].z = 0.5f * (hc[k].z + hc[k].w);
        }
        if (ok) {
            soft_clip_face(hc, g.width, g.height, radius, sc);
            soft_setup(sc, hc, (float)f, g.width, g.height, &r);
        } else {
            atomicOr(err, 8u);
        }
        recs[i] = r;
        cull[i] = cull_setup(r);
    }
    const bool valid = live && r.bx0 <= r.bx1 && r.by0 <= r.by1;
    bin_append(b, g, valid, view, f, r.bx0, r.by0, r.bx1, r.by1, soft_bin_tri(r), blds);
}

// One peel of every item: k_raster_soft_op's resolve and outputs, and, where
// another peel follows, its depth threshold (this layer's shifted depth
// rebuilt from its channels, python/dressi/torch/ops.py:608-615).
// blockIdx.y: the item. neg_inv_radius = -1 / radius.
__global__ __launch_bounds__(64) void k_surface_raster_soft(
        RasterGeom g, const SoftRec* recs, const CullRec* cull, BinBuffers b, float radius,
        float neg_inv_radius, const float* prev, uint32_t layer, uint32_t peels, float4* out,
        float* threshold) {
    const BlockPos blk = block_pos(blockIdx.x, g);
    if (!blk.valid) {
        return;
    }
    const size_t npx = (size_t)g.width * g.height;
    const uint32_t item = blockIdx.y;
    recs += (size_t)item * g.n_faces;
    cull += (size_t)item * g.n_faces;
    prev = prev ? prev + item * npx : nullptr;
    const int lane = threadIdx.x & 63;
    const int px = blk.bx + (lane & 7);
    const int py = blk.by + (lane >> 3);
    const BinView bv = bin_view(b, item * g.n_tiles + blk.tile, g.n_faces);
    __shared__ ResolveLds lds;
    const PixelBest best =
            resolve_block(recs, cull, bv, blk.bx, blk.by, radius, prev, g.width, lds);
    if (px >= (int)g.width || py >= (int)g.height) {
        return;
    }
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    if (best.key != kEmptyKey) {
        const SoftRec& r = recs[key_face(best.key)];
        const float p0 = (float)px + 0.5f;
        const float p1 = (float)py + 0.5f;
        const float dist = signed_dist(p0, p1, r.hx, r.hy, r.ex, r.ey, r.len2);
        o = make_float4(dist, r.fid, hard_z_at(r, p0, p1), 1.f);
    }
    const size_t at = (size_t)py * g.width + px;
    out[((size_t)item * peels + layer) * npx + at] = o;
    if (threshold) {
        const auto clamp01 = [](float x) { return x < 0.f ? 0.f : x > 1.f ? 1.f : x; };
        const float ge = o.x >= 0.f ? 1.f : 0.f;
        const float near = clamp01(o.z) * 0.5f;
        const float far = clamp01(o.x * neg_inv_radius) * 0.5f + 0.5f;
        threshold[item * npx + at] = o.w * (ge * near + (1.f - ge) * far);
    }
}

__global__ void k_soft_clip(const float4* clip, uint32_t n_verts, const float* faces,
                            uint32_t n_faces, uint32_t w, uint32_t h, float radius,
                            uint32_t* err, float4* out) {
    const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= n_faces) {
        return;
    }
    float4 c[3];
    for (int k = 0; k < 3; k++) {
        const uint32_t vi = fid_u(faces[(size_t)f * 3 + k]);
        if (vi >= n_verts) {
            atomicOr(err, 8u);
            return;
        }
        c[k] = clip[vi];
    }
    float4 o[3];
    soft_clip_face(c, w, h, radius, o);
    for (int k = 0; k < 3; k++) {
        out[(size_t)f * 3 + k] = o[k];
    }
}

// z in [-w, w] -> [0, w] per vertex, and the tile counters cleared.
__global__ __launch_bounds__(256) void k_surface_prep(const float4* pos, uint32_t n,
                                                      uint32_t* counts, uint32_t n_counts,
                                                      float4* clip_vk) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        float4 c = pos[i];
        c.z = 0.5f * (c.z + c.w);
        clip_vk[i] = c;
    }
    if (i < n_counts) {
        counts[i] = 0u;
    }
}

}  // namespace dressi

// Scratch of dressi_rasterize_soft_noalloc: one fixed array per GPU (each
// GPU the library runs on holds its own copy until the process ends). In
// host code the name `scratch` is a host-side stand-in, never the device
// array: kernels take the per-device address that hipGetSymbolAddress
// returns (noalloc_scratch below). Every call on a GPU shares that GPU's
// array: host calls are taken one at a time (g_noalloc_mu), calls on one
// stream run in order, and a call on another stream than the GPU's previous
// call first waits for that call's work (an event created with the array's
// address, recorded after every call). A call made while its stream is
// captured into a graph records no wait and no event, so replays of that
// graph race with every other call on the GPU.
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

using namespace dressi;

namespace {

int check_ctx(dressi_ctx* ctx) {
    DRESSI_REQUIRE(ctx != nullptr, "NULL context");
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    return DRESSI_OK;
}

int check_soft_args(const float* soft_clip, const float* face_id, const float* faces_soft,
                    const float* hard_clip, const float* faces_tex, uint32_t width,
                    uint32_t height, float radius_px, const float* out) {
    DRESSI_REQUIRE(soft_clip && face_id && faces_soft && hard_clip && faces_tex && out,
                   "dressi_rasterize_soft: NULL buffer");
    DRESSI_REQUIRE(radius_px > 0.f, "RasterizeSoft: radius_px must be > 0");
    DRESSI_REQUIRE(width > 0 && height > 0, "RasterizeSoft: empty screen");
    return DRESSI_OK;
}

// RasterizeSoft over caller-provided scratch: `recs` / `cull` hold one record
// per face, `bins` fixed_bin_bytes(tiles, kSoftBinCap) bytes (counts cleared
// here by a fill kernel, so the scratch may hold anything on entry).
int launch_rasterize_soft(dressi_ctx* ctx, const RasterGeom& g, const float* soft_clip,
                          const float* face_id, const float* faces_soft, const float* hard_clip,
                          uint32_t n_verts, const float* faces_tex, float radius_px,
                          const float* prev_shifted_depth, SoftRec* recs, void* bins,
                          CullRec* cull, float* out) {
    BinBuffers b;
    fixed_bin_carve(bins, g.n_tiles, kSoftBinCap, &b);
    hipLaunchKernelGGL(k_fill_u32, dim3(div_up(g.n_tiles, 256)), dim3(256), 0, ctx->stream,
                       b.counts, g.n_tiles, 0u);
    DRESSI_CHECK_LAUNCH();
    if (g.n_faces) {
        hipLaunchKernelGGL(k_soft_setup_op, dim3(div_up(g.n_faces, 256)), dim3(256), 0,
                           ctx->stream, g, (const float4*)soft_clip, face_id, faces_soft,
                           (const float4*)hard_clip, n_verts, faces_tex, b, ctx->d_err, recs,
                           cull);
        DRESSI_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_raster_soft_op, dim3(block_grid(g)), dim3(64), 0, ctx->stream, g,
                       (const SoftRec*)recs, (const CullRec*)cull, b, radius_px,
                       prev_shifted_depth, (float4*)out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
char* g_noalloc_ptr[kNoAllocMaxDevices] = {};
hipEvent_t g_noalloc_done[kNoAllocMaxDevices] = {};      // after the GPU's last call
hipStream_t g_noalloc_stream[kNoAllocMaxDevices] = {};   // the stream of that call
bool g_noalloc_used[kNoAllocMaxDevices] = {};

// The device address of this GPU's scratch array, looked up once per device
// with that device current (the caller has made it current), with its
// ordering event; the caller holds g_noalloc_mu.
int noalloc_scratch(int device, char** out) {
    DRESSI_REQUIRE(device >= 0 && device < kNoAllocMaxDevices, "device %d out of range", device);
    if (!g_noalloc_ptr[device]) {
        void* p = nullptr;
        DRESSI_TRY_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        DRESSI_REQUIRE(p != nullptr, "hipGetSymbolAddress returned NULL");
        DRESSI_TRY_HIP(hipEventCreateWithFlags(&g_noalloc_done[device], hipEventDisableTiming));
        g_noalloc_ptr[device] = (char*)p;
    }
    *out = g_noalloc_ptr[device];
    return DRESSI_OK;
}

bool stream_capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

}  // namespace

extern "C" {

int dressi_soft_clip(dressi_ctx* ctx, const float* clip, uint32_t n_verts, const float* faces,
                     uint32_t n_faces, uint32_t width, uint32_t height, float radius_px,
                     float* out) {
    if (int rc = check_ctx(ctx)) return rc;
    DRESSI_REQUIRE(clip && faces && out, "dressi_soft_clip: NULL buffer");
    DRESSI_REQUIRE(radius_px >= 0.f, "SoftClip: radius_px must be >= 0");
    if (n_faces == 0) return DRESSI_OK;
    hipLaunchKernelGGL(k_soft_clip, dim3(div_up(n_faces, 256)), dim3(256), 0, ctx->stream,
                       (const float4*)clip, n_verts, faces, n_faces, width, height, radius_px,
                       ctx->d_err, (float4*)out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_rasterize_soft(dressi_ctx* ctx, const float* soft_clip, const float* face_id,
                          const float* faces_soft, const float* hard_clip, uint32_t n_verts,
                          const float* faces_tex, uint32_t n_faces, uint32_t width,
                          uint32_t height, float radius_px, const float* prev_shifted_depth,
                          float* out) {
    if (int rc = check_ctx(ctx)) return rc;
    if (int rc = check_soft_args(soft_clip, face_id, faces_soft, hard_clip, faces_tex, width,
                                 height, radius_px, out)) return rc;
    const RasterGeom g = make_geom(width, height, 1, n_faces);
    void *recs = nullptr, *bins = nullptr, *cull = nullptr;
    const size_t nf1 = n_faces ? n_faces : 1;
    if (int rc = ctx_workspace(ctx, 0, sizeof(SoftRec) * nf1, &recs)) return rc;
    if (int rc = ctx_workspace(ctx, 1, fixed_bin_bytes(g.n_tiles, kSoftBinCap), &bins)) return rc;
    if (int rc = ctx_workspace(ctx, 3, sizeof(CullRec) * nf1, &cull)) return rc;
    return launch_rasterize_soft(ctx, g, soft_clip, face_id, faces_soft, hard_clip, n_verts,
                                 faces_tex, radius_px, prev_shifted_depth, (SoftRec*)recs, bins,
                                 (CullRec*)cull, out);
}

int dressi_rasterize_soft_noalloc(dressi_ctx* ctx, const float* soft_clip, const float* face_id,
                                  const float* faces_soft, const float* hard_clip,
                                  uint32_t n_verts, const float* faces_tex, uint32_t n_faces,
                                  uint32_t width, uint32_t height, float radius_px,
                                  const float* prev_shifted_depth, float* out) {
    if (int rc = check_ctx(ctx)) return rc;
    if (int rc = check_soft_args(soft_clip, face_id, faces_soft, hard_clip, faces_tex, width,
                                 height, radius_px, out)) return rc;
    const RasterGeom g = make_geom(width, height, 1, n_faces);
    const size_t nf1 = n_faces ? n_faces : 1;
    const size_t rec_bytes = align256(sizeof(SoftRec) * nf1);
    const size_t cull_bytes = align256(sizeof(CullRec) * nf1);
    const size_t bin_bytes_ = fixed_bin_bytes(g.n_tiles, kSoftBinCap);
    const size_t need = rec_bytes + cull_bytes + bin_bytes_;
    DRESSI_REQUIRE(need <= kNoAllocScratchBytes,
                   "dressi_rasterize_soft_noalloc: %u faces on a %ux%u screen need %zu bytes of "
                   "scratch, above the fixed %zu (use dressi_rasterize_soft)",
                   n_faces, width, height, need, kNoAllocScratchBytes);
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    char* base = nullptr;
    if (int rc = noalloc_scratch(ctx->device, &base)) return rc;
    const int dev = ctx->device;
    const bool capturing = stream_capturing(ctx->stream);
    if (!capturing && g_noalloc_used[dev] && g_noalloc_stream[dev] != ctx->stream) {
        DRESSI_TRY_HIP(hipStreamWaitEvent(ctx->stream, g_noalloc_done[dev], 0));
    }
    const int rc = launch_rasterize_soft(ctx, g, soft_clip, face_id, faces_soft, hard_clip,
                                         n_verts, faces_tex, radius_px, prev_shifted_depth,
                                         (SoftRec*)base, base + rec_bytes + cull_bytes,
                                         (CullRec*)(base + rec_bytes), out);
    if (rc == DRESSI_OK && !capturing) {
        DRESSI_TRY_HIP(hipEventRecord(g_noalloc_done[dev], ctx->stream));
        g_noalloc_stream[dev] = ctx->stream;
        g_noalloc_used[dev] = true;
    }
    return rc;
}

// The per-op hard raster's workspaces.
struct HardBins {
    HardRec* recs = nullptr;
    HardBinBuffers b;
};

static int hard_bins(dressi_ctx* ctx, const RasterGeom& g, HardBins* hb) {
    const HardBinSizes z = hard_bin_sizes(g);
    void *recs = nullptr, *bins = nullptr;
    const size_t nf1 = g.n_faces ? g.n_faces : 1;
    if (int rc = ctx_workspace(ctx, 0, sizeof(HardRec) * nf1 * g.n_views, &recs)) return rc;
    if (int rc = ctx_workspace(ctx, 1, z.bytes, &bins)) return rc;
    hb->recs = (HardRec*)recs;
    hard_bin_carve(bins, z, &hb->b);
    return DRESSI_OK;
}

// Setup, binning and raster; hb.b's counters are zero.
static int launch_hard_op(dressi_ctx* ctx, const RasterGeom& g, const HardBins& hb,
                          const float* clip, uint32_t n_verts, const float* faces,
                          const int32_t* faces_i, int gl, const float* attr, uint32_t n_comp,
                          int mode, float* out, size_t attr_view, float* ids,
                          uint32_t n_attr = 1) {
    if (int rc = launch_hard_setup_bin(ctx->stream, g, clip, n_verts, faces, faces_i, gl, hb.b,
                                       ctx->d_err, hb.recs)) return rc;
    return launch_raster_hard(ctx->stream, g, hb.recs, hb.b, attr, n_comp, mode, out, attr_view,
                              ids, n_attr);
}

// `n_items` clip sets [n_items][n_verts] over one face list; attributes
// shared by the items (attr_view 0) or per item (attr_view = n_verts * n_comp
// floats apart); `ids` (optional) gets RasterizeFaceId's output alongside.
static int rasterize_hard_common(dressi_ctx* ctx, const float* clip, uint32_t n_verts,
                                 const float* attr, uint32_t n_comp, const float* faces,
                                 uint32_t n_faces, uint32_t width, uint32_t height, int mode,
                                 float* out, uint32_t n_items = 1, size_t attr_view = 0,
                                 float* ids = nullptr) {
    if (int rc = check_ctx(ctx)) return rc;
    DRESSI_REQUIRE(clip && (faces || n_faces == 0) && out && (mode == 1 || attr),
                   "rasterize: NULL buffer");
    DRESSI_REQUIRE(width > 0 && height > 0, "rasterize: empty screen");
    DRESSI_REQUIRE(mode == 1 || (n_comp >= 1 && n_comp <= 4), "rasterize: n_comp must be 1..4");
    DRESSI_REQUIRE(n_items >= 1 && (uint64_t)n_items * n_faces < (1ull << 31) &&
                           (uint64_t)n_items * n_verts < (1ull << 31),
                   "rasterize: too many items");
    const RasterGeom g = make_geom(width, height, n_items, n_faces);
    HardBins hb;
    if (int rc = hard_bins(ctx, g, &hb)) return rc;
    if (int rc = launch_zero(ctx->stream, hb.b.counts, hb.b.clear_bytes()))
        return rc;
    return launch_hard_op(ctx, g, hb, clip, n_verts, faces, nullptr, 0, attr,
                          mode == 1 ? 1 : n_comp, mode, out, attr_view, ids);
}

int dressi_rasterize(dressi_ctx* ctx, const float* clip, uint32_t n_verts, const float* attr,
                     uint32_t n_comp, const float* faces, uint32_t n_faces, uint32_t width,
                     uint32_t height, float* out) {
    return rasterize_hard_common(ctx, clip, n_verts, attr, n_comp, faces, n_faces, width,
                                 height, 0, out);
}

int dressi_rasterize_face_id(dressi_ctx* ctx, const float* clip, uint32_t n_verts,
                             const float* faces, uint32_t n_faces, uint32_t width,
                             uint32_t height, float* out) {
    return rasterize_hard_common(ctx, clip, n_verts, nullptr, 1, faces, n_faces, width, height,
                                 1, out);
}

int dressi_rasterize_batch(dressi_ctx* ctx, const float* clip, uint32_t n_verts,
                           uint32_t n_items, const float* attr, uint32_t n_comp,
                           int attr_per_item, const float* faces, uint32_t n_faces,
                           uint32_t width, uint32_t height, float* out, float* face_id) {
    return rasterize_hard_common(ctx, clip, n_verts, attr, n_comp, faces, n_faces, width, height,
                                 0, out, n_items, attr_per_item ? (size_t)n_verts * n_comp : 0,
                                 face_id);
}

// The torch surface's rasterize: pos {N,V} VEC4 clip positions with z in
// [-w, w]; clip_vk gets them with z remapped to [0, w], rast {N,H,W} VEC4 the
// winner's (u, v, z / w, face + 1).
int dressi_surface_rasterize(dressi_ctx* ctx, const float* pos, uint32_t n_verts,
                             uint32_t n_items, const int32_t* faces, uint32_t n_faces,
                             uint32_t width, uint32_t height, float* clip_vk, float* rast) {
    if (int rc = check_ctx(ctx)) return rc;
    DRESSI_REQUIRE((pos || n_verts == 0) && (faces || n_faces == 0) &&
                           (clip_vk || n_verts == 0) && rast,
                   "rasterize: NULL buffer");
    DRESSI_REQUIRE(width > 0 && height > 0, "rasterize: empty screen");
    DRESSI_REQUIRE(n_items >= 1 && (uint64_t)n_items * n_faces < (1ull << 31) &&
                           (uint64_t)n_items * n_verts < (1ull << 31),
                   "rasterize: too many items");
    const RasterGeom g = make_geom(width, height, n_items, n_faces);
    HardBins hb;
    if (int rc = hard_bins(ctx, g, &hb)) return rc;
    const uint32_t n_clear = (uint32_t)(hb.b.clear_bytes() / sizeof(uint32_t));
    const uint32_t n_prep = std::max(n_verts * n_items, n_clear);
    hipLaunchKernelGGL(k_surface_prep, dim3(div_up(n_prep, 256)), dim3(256), 0, ctx->stream,
                       (const float4*)pos, n_verts * n_items, hb.b.counts, n_clear,
                       (float4*)clip_vk);
    DRESSI_CHECK_LAUNCH();
    return launch_hard_op(ctx, g, hb, pos, n_verts, nullptr, faces, 1, pos, 4, 2, rast,
                          (size_t)n_verts * 4, nullptr);
}

// The torch surface's rasterize_soft: pos {N,V} VEC4, z in [-w, w] -> out
// {N,K,H,W} VEC4. Items go through in groups whose bins fit kSoftGroupBytes.
int dressi_surface_rasterize_soft(dressi_ctx* ctx, const float* pos, uint32_t n_verts,
                                  uint32_t n_items, const float* faces, uint32_t n_faces,
                                  uint32_t width, uint32_t height, float radius_px,
                                  float neg_inv_radius, uint32_t peels, float* threshold,
                                  float* out) {
    constexpr size_t kSoftGroupBytes = (size_t)256 << 20;
    if (int rc = check_ctx(ctx)) return rc;
    DRESSI_REQUIRE((pos || n_verts == 0) && (faces || n_faces == 0) && out &&
                           (threshold || peels == 1),
                   "rasterize_soft: NULL buffer");
    DRESSI_REQUIRE(radius_px > 0.f, "RasterizeSoft: radius_px must be > 0");
    DRESSI_REQUIRE(width > 0 && height > 0, "RasterizeSoft: empty screen");
    DRESSI_REQUIRE(peels >= 1, "RasterizeSoft: peels must be >= 1");
    if (n_items == 0) return DRESSI_OK;
    const size_t npx = (size_t)width * height;
    const size_t item_bytes = fixed_bin_bytes(make_geom(width, height, 1, n_faces).n_tiles,
                                              kSoftBinCap);
    uint32_t group = (uint32_t)std::min<size_t>(
            std::max<size_t>(kSoftGroupBytes / item_bytes, 1), n_items);
    group = std::min(group, kMaxBatchItems);
    while (group > 1 && (uint64_t)group * n_faces >= (1ull << 31)) group /= 2;
    for (uint32_t i0 = 0; i0 < n_items; i0 += group) {
        const uint32_t n = std::min(group, n_items - i0);
        const RasterGeom g = make_geom(width, height, n, n_faces);
        // (the raster takes an item on the grid's y: tiles of one view)
        const RasterGeom g1 = make_geom(width, height, 1, n_faces);
        void *recs = nullptr, *bins = nullptr, *cull = nullptr;
        const size_t nf = (size_t)(n_faces ? n_faces : 1) * n;
        if (int rc = ctx_workspace(ctx, 0, sizeof(SoftRec) * nf, &recs)) return rc;
        if (int rc = ctx_workspace(ctx, 1, fixed_bin_bytes(g.n_tiles * n, kSoftBinCap), &bins))
            return rc;
        if (int rc = ctx_workspace(ctx, 3, sizeof(CullRec) * nf, &cull)) return rc;
        BinBuffers b;
        fixed_bin_carve(bins, g.n_tiles * n, kSoftBinCap, &b);
        if (int rc = launch_zero(ctx->stream, b.counts, sizeof(uint32_t) * g.n_tiles * n))
            return rc;
        const float* p = pos + (size_t)i0 * n_verts * 4;
        if (n_faces) {
            hipLaunchKernelGGL(k_surface_soft_setup, dim3(div_up(n * n_faces, 256)), dim3(256), 0,
                               ctx->stream, g, (const float4*)p, n_verts, faces, radius_px, b,
                               ctx->d_err, (SoftRec*)recs, (CullRec*)cull);
            DRESSI_CHECK_LAUNCH();
        }
        for (uint32_t k = 0; k < peels; k++) {
            // layer k reads layer k - 1's threshold and writes its own over it
            // (each pixel its own)
            float* thr = threshold ? threshold + i0 * npx : nullptr;
            hipLaunchKernelGGL(k_surface_raster_soft, dim3(block_grid(g1), n), dim3(64), 0,
                               ctx->stream, g1, (const SoftRec*)recs, (const CullRec*)cull, b,
                               radius_px, neg_inv_radius, k ? thr : (const float*)nullptr, k, peels,
                               (float4*)out + (size_t)i0 * peels * npx,
                               k + 1 < peels ? thr : nullptr);
            DRESSI_CHECK_LAUNCH();
        }
    }
    return DRESSI_OK;
}

}  // extern "C"

namespace dressi {

int raster_attrs(dressi_ctx* ctx, const float* clip, uint32_t n_verts, uint32_t n_views,
                 const float* attr, uint32_t n_attr, const float* faces, uint32_t n_faces,
                 uint32_t width, uint32_t height, float* out) {
    const RasterGeom g = make_geom(width, height, n_views, n_faces);
    HardBins hb;
    if (int rc = hard_bins(ctx, g, &hb)) return rc;
    if (int rc = launch_zero(ctx->stream, hb.b.counts, hb.b.clear_bytes()))
        return rc;
    return launch_hard_op(ctx, g, hb, clip, n_verts, faces, nullptr, 0, attr, 4, 0, out,
                          (size_t)n_verts * 4, nullptr, n_views > 1 ? 1 : n_attr);
}

}  // namespace dressi
