// ibl.hip -- the split-sum IBL ops as per-op entry points (reference
// layouts): EquirectSample and its map VJP, AvgPool2x2 and its VJP,
// IrradianceConv / PrefilterConv and their transposes, PrefilterEnv and
// BrdfIntegrationLut (src/core/f_ops.cpp:2785-3415, src/core/ibl_math.h).
//
// The dense convolutions add each output texel's terms in the reference's
// loop order, so with the reference's direction tables (ibl_core.h) their
// sums are the reference's bit for bit. The map
// VJP of EquirectSample scatters in 64-bit fixed point (exact, so the
// result does not depend on the order of the atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "dressi_hip.h"
#include "ibl_core.h"
#include "internal.h"

namespace dressi {
namespace {

// ---------------------------------------------------------------------------
// EquirectSample
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_eq_sample(const float* map, int mw, int mh, uint32_t n,
                                                   const float* dir, size_t npx, float* out) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npx) {
        return;
    }
    float u, v;
    float res[4] = {0.f, 0.f, 0.f, 0.f};
    if (dir_to_equirect(mk3(dir[p * 3 + 0], dir[p * 3 + 1], dir[p * 3 + 2]), &u, &v)) {
        taps_fetch(taps_wrap(mw, mh, u, v), map, n, res);
    }
    for (uint32_t c = 0; c < n; c++) {
        out[p * n + c] = res[c];
    }
}

// Map VJP of EquirectSample (EquirectSampleBwd, f_ops.cpp:2823-2919): each
// pixel's gy * tap weight (the reference's float product) is added to its
// four texels in 64-bit fixed point, so any grouping of the adds gives the
// same bits.
//
// What bounded the plain form (one global atomic per pixel, tap and channel)
// was the atomics themselves: neighbouring pixels look at the same few
// texels, and adds to one line follow each other at ~15 ns (512 x 512
// pixels, 3 channels: 18.7 ms onto a 4 x 2 map, 1.6 ms onto 32 x 16, 0.9 ms
// onto 128 x 64). Here a workgroup sums a tile of 1024 pixels in LDS and
// sends each touched texel to memory once. The LDS adds of one wave to the
// same texel follow each other as well (20-25 us on each of these maps with
// one sum per texel and 256 threads), so a texel has up to 32 sums side by
// side, each taking every such lane's adds: 9.4-15 us.
constexpr uint32_t kScatterPixels = 1024;
constexpr uint32_t kScatterThreads = 1024;
// Sums per texel in the hash table (2^kScatterHashCopies).
constexpr uint32_t kScatterHashCopies = 2;
// Entries (texel, channel) up to which a workgroup keeps the whole map in
// LDS (48 KB: two workgroups of 16 waves fill a CU's 32, so that LDS up to 80
// KB each costs none); above it a hash table of the texels that the tile
// touches (at most 56 KB; a tile of a coherent direction image touches tens to
// hundreds). A few tiles of incoherent directions on a large map are slower so
// than the plain form, by the probing of one tile (1000 onto 512 x 256: 27 ->
// 34 us).
constexpr uint32_t kScatterDirect = 6144;
constexpr uint32_t kScatterEmpty = 0xffffffffu;
constexpr uint32_t kScatterProbes = 8;
inline uint32_t scatter_slots_log2(uint32_t n) { return n == 4 ? 10u : 11u; }
// Workgroups (and partial maxima) of the preparation.
constexpr uint32_t kScatterParts = 256;

// max |gy| as float bits (non-negative floats order like their bits; inf and
// NaN do not count), one partial per workgroup, and the cleared accumulators
__global__ __launch_bounds__(256) void k_eq_scatter_prep(const float* x, size_t count,
                                                         uint32_t* part,
                                                         unsigned long long* acc, size_t n_acc) {
    __shared__ uint32_t wmax[4];
    const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t step = (size_t)gridDim.x * blockDim.x;
    for (size_t i = t0; i < n_acc; i += step) {
        acc[i] = 0ull;
    }
    uint32_t m = 0;
    for (size_t i = t0; i < count; i += step) {
        const uint32_t b = __float_as_uint(fabsf(x[i]));
        m = b > m && b < 0x7f800000u ? b : m;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)m, o);
        m = other > m ? other : m;
    }
    if ((threadIdx.x & 63) == 0) {
        wmax[threadIdx.x >> 6] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; k++) {
            m = wmax[k] > m ? wmax[k] : m;
        }
        part[blockIdx.x] = m;
    }
}

// The largest of the partial maxima (n_part <= 256 <= the workgroup's size).
__device__ __forceinline__ uint32_t scatter_max(const uint32_t* part, uint32_t n_part,
                                                uint32_t* wmax) {
    uint32_t m = threadIdx.x < n_part ? part[threadIdx.x] : 0u;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)m, o);
        m = other > m ? other : m;
    }
    if (threadIdx.x < 256 && (threadIdx.x & 63) == 0) {
        wmax[threadIdx.x >> 6] = m;
    }
    __syncthreads();
    m = wmax[0];
    for (int k = 1; k < 4; k++) {
        m = wmax[k] > m ? wmax[k] : m;
    }
    return m;
}

// Fixed-point exponent for sums bounded by max|x| * count: every partial
// sum stays below 2^62 in magnitude.
__device__ __forceinline__ int fixed_exponent(uint32_t max_bits, double count) {
    const double bound = (double)__uint_as_float(max_bits) * count;
    if (!(bound > 0.0)) {
        return 0;
    }
    int e;
    frexp(bound, &e);  // bound < 2^e
    return 62 - e;
}

// One workgroup per tile of tile_w x (1024 / tile_w) pixels, a thread per
// pixel. `slots_log2`: 0 = the whole map in LDS, else the hash table's size.
// 2^copies_log2 sums per texel (and channel), neighbours in LDS: a lane adds
// to the one of its number. The launch's tiles begin at `tile0`.
__global__ __launch_bounds__(kScatterThreads) void k_eq_scatter(
        const float* gy, uint32_t n, const float* dir, uint32_t dw, uint32_t dh, uint32_t tile_w,
        uint32_t tiles_x, int mw, int mh, const uint32_t* part, uint32_t n_part,
        uint32_t slots_log2, uint32_t copies_log2, uint32_t tile0, unsigned long long* acc) {
    extern __shared__ unsigned long long lds[];
    __shared__ uint32_t wmax[4];
    const uint32_t tid = threadIdx.x;
    const uint32_t slots = 1u << slots_log2;
    const uint32_t n_sum = slots_log2 ? slots * n : (uint32_t)(mw * mh) * n;
    uint32_t* keys = (uint32_t*)(lds + ((size_t)n_sum << copies_log2));  // hash table only
    for (uint32_t i = tid; i < n_sum << copies_log2; i += kScatterThreads) {
        lds[i] = 0ull;
    }
    if (slots_log2) {
        for (uint32_t i = tid; i < slots; i += kScatterThreads) {
            keys[i] = kScatterEmpty;
        }
    }
    const uint32_t tile = tile0 + blockIdx.x;
    const uint32_t x = (tile % tiles_x) * tile_w + tid % tile_w;
    const uint32_t y = (tile / tiles_x) * (kScatterPixels / tile_w) + tid / tile_w;
    const uint32_t copy = tid & ((1u << copies_log2) - 1u);
    const int k = fixed_exponent(scatter_max(part, n_part, wmax), (double)((size_t)dw * dh));
    __syncthreads();
    const size_t p = (size_t)y * dw + x;
    float u, v;
    if (x < dw && y < dh &&
        dir_to_equirect(mk3(dir[p * 3 + 0], dir[p * 3 + 1], dir[p * 3 + 2]), &u, &v)) {
        const Taps t = taps_wrap(mw, mh, u, v);
        float g[4];
        for (uint32_t c = 0; c < n; c++) {
            g[c] = gy[p * n + c];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t texel = (uint32_t)t.idx[j];
            uint32_t at = texel;
            bool in_lds = true;
            if (slots_log2) {
                at = (texel * 2654435761u) >> (32 - slots_log2);
                in_lds = false;
                for (uint32_t tries = 0; tries < kScatterProbes; tries++) {
                    uint32_t key = __hip_atomic_load(&keys[at], __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (key == kScatterEmpty) {
                        key = atomicCAS(&keys[at], kScatterEmpty, texel);
                        key = key == kScatterEmpty ? texel : key;
                    }
                    if (key == texel) {
                        in_lds = true;
                        break;
                    }
                    at = (at + 1) & (slots - 1);
                }
            }
            for (uint32_t c = 0; c < n; c++) {
                const float prod = g[c] * t.w[j];
                const long long fx = __double2ll_rn(ldexp((double)prod, k));
                if (!fx) {
                    continue;
                }
                if (in_lds) {
                    atomicAdd(&lds[((at * n + c) << copies_log2) + copy],
                              (unsigned long long)fx);
                } else {
                    atomicAdd(&acc[(size_t)texel * n + c], (unsigned long long)fx);
                }
            }
        }
    }
    __syncthreads();
    // a lane per sum; a texel's lanes meet by shuffles
    const uint32_t n_all = n_sum << copies_log2;
    for (uint32_t i0 = 0; i0 < n_all; i0 += kScatterThreads) {
        const uint32_t i = i0 + tid;
        unsigned long long a = i < n_all ? lds[i] : 0ull;
        for (uint32_t o = 1u << copies_log2 >> 1; o >= 1; o >>= 1) {
            a += (unsigned long long)__shfl_xor((long long)a, (int)o);
        }
        const uint32_t s = i >> copies_log2;
        if (a && copy == 0) {
            const size_t texel = slots_log2 ? keys[s / n] : s / n;
            atomicAdd(&acc[texel * n + s % n], a);
        }
    }
}

__global__ __launch_bounds__(256) void k_fixed_resolve(const unsigned long long* acc,
                                                       size_t count, const uint32_t* part,
                                                       uint32_t n_part, double npx, float* out) {
    __shared__ uint32_t wmax[4];
    const int k = fixed_exponent(scatter_max(part, n_part, wmax), npx);
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        out[i] = (float)ldexp((double)(long long)acc[i], -k);
    }
}

// ---------------------------------------------------------------------------
// AvgPool2x2 (Reduce2x2Sum * 0.25, f_ops.cpp:996-1033, 3411-3415)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_pool_fwd(const float* x, int w, int h, uint32_t n,
                                                  int ow, int oh, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ow * oh) {
        return;
    }
    const int ox = i % ow, oy = i / ow;
    for (uint32_t c = 0; c < n; c++) {
        float acc = 0.f;
        for (int dy = 0; dy < 2; dy++) {
            for (int dx = 0; dx < 2; dx++) {
                const int px = 2 * ox + dx, py = 2 * oy + dy;
                if (px < w && py < h) {
                    acc += x[((size_t)py * w + px) * n + c];
                }
            }
        }
        out[(size_t)i * n + c] = acc * 0.25f;
    }
}

// VJP: UpsampleNearest2x(gy * 0.25) (f_ops.cpp:958-994)
__global__ __launch_bounds__(256) void k_pool_bwd(const float* gy, int w, int h, uint32_t n,
                                                  int ow, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w * h) {
        return;
    }
    const int px = i % w, py = i / w;
    for (uint32_t c = 0; c < n; c++) {
        out[(size_t)i * n + c] = gy[((size_t)(py / 2) * ow + px / 2) * n + c] * 0.25f;
    }
}

// ---------------------------------------------------------------------------
// Dense equirect convolutions
// ---------------------------------------------------------------------------

enum ConvMode : int {
    kIrrFwd = 0,   // out(t) = scale * sum_s e(s) max(N_t . d_s, 0) sin_s
    kIrrBwd = 1,   // out(s) = scale * sum_t gy(t) max(N_t . d_s, 0) sin_s
    kPrefNorm = 2, // out(t) = sum_s ggx(r_t . d_s) sin_s
    kPrefFwd = 3,  // out(t) = sum_s e(s) ggx(r_t . d_s) sin_s / max(W_t, 1e-12)
    kPrefBwd = 4,  // out(s) = sin_s sum_t gy(t) ggx(r_t . d_s) / max(W_t, 1e-12)
};

// Each output texel's sum runs over the other side in the reference's loop
// order (f_ops.cpp:2970-3087, 3166-3348), one float add after the other, so
// the terms can be formed in parallel but not added so. A workgroup takes
// kConvOut outputs: four waves form the terms (weight times value, one
// rounding each, as the reference) of a chunk of kConvChunk sources into one
// LDS buffer while the fifth adds the chunk before from the other, one lane
// per output and channel, in order.
//
// One thread per output that did both (the form before) had 8192 / 64 waves
// and less, each at the latency of a weight, a load and an add per source:
// 2.4-3.2 ms from an 8192-texel source whatever the output's size. Now
// 128 x 64 from 128 x 64 takes 64 us (67 M weights of ~40 VALU instructions:
// issue), its transpose 86 us (one division more). Few outputs have the form
// below.
constexpr uint32_t kConvOut = 8;
constexpr uint32_t kConvChunk = 128;
// A row of terms, padded so that the adding lanes' 16-byte reads start 4
// banks apart.
constexpr uint32_t kConvRow = kConvChunk + 4;
constexpr uint32_t kConvThreads = 5 * 64;

// The weight of an output and a source (`nj`: PrefBwd's normaliser).
template <int MODE>
__device__ __forceinline__ float conv_weight(float dt, float sin_s, float nj, float alpha,
                                             bool* used) {
    if (MODE == kIrrFwd || MODE == kIrrBwd) {
        return (dt > 0.f ? dt : 0.f) * sin_s;
    }
    const float w = ggx_conv_weight(dt, alpha);
    if (MODE == kPrefNorm || MODE == kPrefFwd) {
        return w * sin_s;
    }
    *used = *used && !(w <= 0.f);  // the reference skips these
    return w / nj;
}

template <int MODE>
__device__ __forceinline__ float conv_result(float sum, float scale, float norm, float sin_i) {
    if (MODE == kIrrFwd || MODE == kIrrBwd) {
        return sum * scale;
    }
    if (MODE == kPrefFwd) {
        return sum / (norm > 1e-12f ? norm : 1e-12f);
    }
    return MODE == kPrefBwd ? sum * sin_i : sum;
}

// `odir` are the output-map directions, `sdir` the source (env) directions;
// `in` is the env (forward modes) or the output-map gradient (backward
// modes), N channels. The launch's outputs begin at `first`.
template <int MODE, int N>
__global__ __launch_bounds__(kConvThreads) void k_eq_conv(const float4* odir, uint32_t n_o,
                                                          const float4* sdir, uint32_t n_s,
                                                          const float* in, const float* norm,
                                                          float alpha, float scale,
                                                          uint32_t first, float* out) {
    constexpr bool kBwd = MODE == kIrrBwd || MODE == kPrefBwd;
    __shared__ alignas(16) float term[2][kConvOut][N][kConvRow];
    const uint32_t n_i = kBwd ? n_s : n_o;
    const uint32_t n_j = kBwd ? n_o : n_s;
    const float4* idir = kBwd ? sdir : odir;
    const float4* jdir = kBwd ? odir : sdir;
    const uint32_t i0 = first + blockIdx.x * kConvOut;
    const uint32_t n_chunks = (n_j + kConvChunk - 1) / kConvChunk;
    const uint32_t tid = threadIdx.x;
    const bool adds = tid >= 256;  // the fifth wave

    // forming: one source per thread, every second output (two waves take the
    // even ones, so an output's direction is the wave's: scalar loads)
    const uint32_t src = tid & (kConvChunk - 1);
    const uint32_t half = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 7)) & 1u;
    float4 me[kConvOut / 2];
#pragma unroll
    for (uint32_t o = 0; o < kConvOut / 2; o++) {
        const uint32_t i = i0 + 2 * o + half;
        me[o] = idir[i < n_i ? i : n_i - 1];
    }
    struct Source {
        float4 d;
        float norm, val[N];
    };
    const auto load = [&](uint32_t chunk, Source* s) {
        const uint32_t j = chunk * kConvChunk + src;
        const uint32_t jc = j < n_j ? j : n_j - 1;
        s->d = jdir[jc];
        if (MODE == kPrefBwd) {
            s->norm = norm[jc];
        }
        if (MODE != kPrefNorm) {
#pragma unroll
            for (int c = 0; c < N; c++) {
                s->val[c] = in[(size_t)jc * N + c];
            }
        }
    };
    // a term past the last source is +0: a sum that starts at +0 is never -0,
    // so adding +0 leaves it as it is
    const auto form = [&](uint32_t chunk, const Source& s) {
        const float nj = MODE == kPrefBwd && s.norm > 1e-12f ? s.norm : 1e-12f;
        const bool live = chunk * kConvChunk + src < n_j;
#pragma unroll
        for (uint32_t o = 0; o < kConvOut / 2; o++) {
            const float4 ot = kBwd ? s.d : me[o];
            const float4 sd = kBwd ? me[o] : s.d;
            const float dt = ot.x * sd.x + ot.y * sd.y + ot.z * sd.z;
            bool used = live;
            const float w = conv_weight<MODE>(dt, sd.w, nj, alpha, &used);
            float(*row)[kConvRow] = term[chunk & 1u][2 * o + half];
            if (MODE == kPrefNorm) {
                row[0][src] = used ? w : 0.f;
            } else {
#pragma unroll
                for (int c = 0; c < N; c++) {
                    row[c][src] = used ? s.val[c] * w : 0.f;
                }
            }
        }
    };

    const uint32_t lane = tid & 63u;
    const bool sums = adds && lane < kConvOut * N;
    const uint32_t so = lane / N, sc = lane % N;
    float acc = 0.f;
    Source cur{}, next{};
    if (!adds) {
        load(0, &cur);
        load(n_chunks > 1 ? 1 : 0, &next);
        form(0, cur);
        cur = next;
    }
    __syncthreads();
    for (uint32_t chunk = 0; chunk < n_chunks; chunk++) {
        if (!adds) {
            if (chunk + 1 < n_chunks) {
                load(chunk + 2 < n_chunks ? chunk + 2 : chunk + 1, &next);
                form(chunk + 1, cur);
                cur = next;
            }
        } else if (sums) {
            // the next 16 terms' reads in flight while these 16 are added
            const float4* t = (const float4*)term[chunk & 1u][so][sc];
            float4 now[4], next[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                now[k] = t[k];
            }
#pragma unroll
            for (uint32_t q = 4; q <= kConvChunk / 4; q += 4) {
                if (q < kConvChunk / 4) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        next[k] = t[q + k];
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    acc += now[k].x;
                    acc += now[k].y;
                    acc += now[k].z;
                    acc += now[k].w;
                    now[k] = next[k];
                }
            }
        }
        __syncthreads();
    }
    const uint32_t i = i0 + so;
    if (!sums || i >= n_i) {
        return;
    }
    out[(size_t)i * N + sc] = conv_result<MODE>(acc, scale, MODE == kPrefFwd ? norm[i] : 0.f,
                                                MODE == kPrefBwd ? idir[i].w : 0.f);
}

// The same sums for few outputs, where the chain of adds bounds (4.7 cycles
// each by itself, 17 us for 8192). Four outputs to a workgroup, 256 sources a
// chunk, three buffers: the adding wave starts a chunk's reads before it has
// added the one before, and the forming waves' loads are up to four chunks
// ahead and stay in flight across the barriers, which wait for LDS alone.
// From an 8192-texel source 1 to 512 outputs take 27 us and 2048 take 30,
// where the form above takes 37-41 and 43 (its adding wave waits for each
// chunk's first reads, and its chunks for the loads of the next). Chunks of
// 128 here 32-34 us, 16 reads in flight 33. From 8192 outputs the weights
// bound and three buffers' LDS costs waves: 64 us above, 74 with them.
constexpr uint32_t kFewMax = 2048;
constexpr uint32_t kFewOut = 4;
constexpr uint32_t kFewChunk = 256;
constexpr uint32_t kFewRow = kFewChunk + 4;
constexpr uint32_t kFewLoads = 4;  // chunks whose sources are on their way
constexpr int kFewAhead = 8;        // the adding wave's 16-byte reads in flight

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int MODE, int N>
__global__ __launch_bounds__(kConvThreads) void k_eq_conv_few(const float4* odir, uint32_t n_o,
                                                              const float4* sdir, uint32_t n_s,
                                                              const float* in, const float* norm,
                                                              float alpha, float scale,
                                                              uint32_t first, float* out) {
    constexpr bool kBwd = MODE == kIrrBwd || MODE == kPrefBwd;
    __shared__ alignas(16) float term[3][kFewOut][N][kFewRow];
    const uint32_t n_i = kBwd ? n_s : n_o;
    const uint32_t n_j = kBwd ? n_o : n_s;
    const float4* idir = kBwd ? sdir : odir;
    const float4* jdir = kBwd ? odir : sdir;
    const uint32_t i0 = first + blockIdx.x * kFewOut;
    const uint32_t n_chunks = (n_j + kFewChunk - 1) / kFewChunk;
    const uint32_t src = threadIdx.x;
    if (src < 256) {
        float4 me[kFewOut];
#pragma unroll
        for (uint32_t o = 0; o < kFewOut; o++) {
            const uint32_t i = i0 + o;
            me[o] = idir[i < n_i ? i : n_i - 1];
        }
        struct Source {
            float4 d;
            float norm, val[N];
        } s[kFewLoads];
        const auto load = [&](uint32_t chunk, Source* to) {
            const uint32_t j = (chunk < n_chunks ? chunk : n_chunks - 1) * kFewChunk + src;
            const uint32_t jc = j < n_j ? j : n_j - 1;
            to->d = jdir[jc];
            if (MODE == kPrefBwd) {
                to->norm = norm[jc];
            }
            if (MODE != kPrefNorm) {
#pragma unroll
                for (int c = 0; c < N; c++) {
                    to->val[c] = in[(size_t)jc * N + c];
                }
            }
        };
#pragma unroll
        for (uint32_t k = 0; k < kFewLoads; k++) {
            load(k, &s[k]);
        }
        // Chunk c is formed before barrier c, its first terms are read after
        // barrier c, the others after barrier c + 1, and its buffer is free
        // after barrier c + 2. Two chunks too many, +0 terms that no sum
        // takes: without a branch around the loads the waits are for one
        // chunk's.
        uint32_t buf = 0;
        for (uint32_t c0 = 0;; c0 += kFewLoads) {
#pragma unroll
            for (uint32_t k = 0; k < kFewLoads; k++) {
                const uint32_t c = c0 + k;
                const float nj = MODE == kPrefBwd && s[k].norm > 1e-12f ? s[k].norm : 1e-12f;
#pragma unroll
                for (uint32_t o = 0; o < kFewOut; o++) {
                    const float4 ot = kBwd ? s[k].d : me[o];
                    const float4 sd = kBwd ? me[o] : s[k].d;
                    const float dt = ot.x * sd.x + ot.y * sd.y + ot.z * sd.z;
                    bool used = c * kFewChunk + src < n_j;
                    const float w = conv_weight<MODE>(dt, sd.w, nj, alpha, &used);
#pragma unroll
                    for (int ch = 0; ch < N; ch++) {
                        const float x = MODE == kPrefNorm ? w : s[k].val[ch] * w;
                        term[buf][o][ch][src] = used ? x : 0.f;
                    }
                }
                load(c + kFewLoads, &s[k]);
                lds_barrier();
                if (c > n_chunks) {
                    return;
                }
                buf = buf == 2 ? 0 : buf + 1;
            }
        }
    }
    const uint32_t lane = src & 63u;
    const bool sums = lane < kFewOut * N;
    const uint32_t so = sums ? lane / N : 0u, sc = sums ? lane % N : 0u;
    __builtin_amdgcn_s_setprio(3);
    float acc = 0.f;
    float4 a[kFewAhead], b[kFewAhead];
    const auto add = [&](const float4* x) {
#pragma unroll
        for (int k = 0; k < kFewAhead; k++) {
            acc += x[k].x;
            acc += x[k].y;
            acc += x[k].z;
            acc += x[k].w;
        }
    };
    lds_barrier();
    lds_barrier();
#pragma unroll
    for (int k = 0; k < kFewAhead; k++) {
        a[k] = ((const float4*)term[0][so][sc])[k];
    }
    uint32_t buf = 0;
    for (uint32_t chunk = 0; chunk < n_chunks; chunk++) {
        const float4* t = (const float4*)term[buf][so][sc];
        buf = buf == 2 ? 0 : buf + 1;
        // formed before the last barrier (after the last chunk: +0 terms)
        const float4* t_next = (const float4*)term[buf][so][sc];
#pragma unroll
        for (int q = 0; q < (int)kFewChunk / 4; q += 2 * kFewAhead) {
#pragma unroll
            for (int k = 0; k < kFewAhead; k++) {
                b[k] = t[q + kFewAhead + k];
            }
            add(a);
#pragma unroll
            for (int k = 0; k < kFewAhead; k++) {
                a[k] = q + 2 * kFewAhead < (int)kFewChunk / 4 ? t[q + 2 * kFewAhead + k]
                                                              : t_next[k];
            }
            add(b);
        }
        lds_barrier();
    }
    const uint32_t i = i0 + so;
    if (sums && i < n_i) {
        out[(size_t)i * N + sc] = conv_result<MODE>(acc, scale, MODE == kPrefFwd ? norm[i] : 0.f,
                                                    MODE == kPrefBwd ? idir[i].w : 0.f);
    }
}

// PrefilterEnv (f_ops.cpp:3089-3157): per output texel, n_samples GGX
// importance samples (Hammersley table), NoL-weighted bilinear taps.
__global__ __launch_bounds__(64) void k_prefilter_env(const float4* odir, uint32_t n_o,
                                                      const float* env, int sw, int sh,
                                                      uint32_t n, const float4* smp,
                                                      uint32_t n_samples, float roughness,
                                                      float* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_o) {
        return;
    }
    const float4 o = odir[i];
    const V3f N = mk3(o.x, o.y, o.z);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    float wsum = 0.f;
    for (uint32_t s = 0; s < n_samples; s++) {
        const V3f h = importance_sample_ggx(smp[s], roughness, N);
        const float ndh2 = 2.f * dot3(N, h);
        const V3f l = normalize3(mk3(ndh2 * h.x - N.x, ndh2 * h.y - N.y, ndh2 * h.z - N.z));
        const float nol = dot3(N, l);
        if (nol > 0.f) {
            float u, v, tap[4];
            equirect_uv(l, &u, &v);
            taps_fetch(taps_wrap(sw, sh, u, v), env, n, tap);
            for (uint32_t c = 0; c < n; c++) {
                acc[c] += tap[c] * nol;
            }
            wsum += nol;
        }
    }
    const float wden = wsum > 1e-4f ? wsum : 1e-4f;
    for (uint32_t c = 0; c < n; c++) {
        out[(size_t)i * n + c] = acc[c] / wden;
    }
}

// BrdfIntegrationLut (f_ops.cpp:3350-3409)
__global__ __launch_bounds__(64) void k_brdf_lut(int w, int h, const float4* smp,
                                                 uint32_t n_samples, float2* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w * h) {
        return;
    }
    const int ox = i % w, oy = i / w;
    const float rough = ((float)oy + 0.5f) / (float)h;
    const float k = rough * rough / 2.f;
    const float ndv = ((float)ox + 0.5f) / (float)w;
    const float s0 = 1.f - ndv * ndv;
    const V3f V = mk3(sqrtf(s0 > 0.f ? s0 : 0.f), 0.f, ndv);
    float a = 0.f, b = 0.f;
    for (uint32_t s = 0; s < n_samples; s++) {
        const V3f hv = importance_sample_ggx(smp[s], rough, mk3(0.f, 0.f, 1.f));
        const float vdh2 = 2.f * dot3(V, hv);
        const V3f l = normalize3(mk3(vdh2 * hv.x - V.x, vdh2 * hv.y - V.y, vdh2 * hv.z - V.z));
        const float nol = l.z > 0.f ? l.z : 0.f;
        const float noh = hv.z > 0.f ? hv.z : 0.f;
        const float vd = dot3(V, hv);
        const float voh = vd > 0.f ? vd : 0.f;
        if (nol > 0.f) {
            const float g = g1_ibl(ndv, k) * g1_ibl(nol, k);
            const float nd = noh * ndv;
            const float gv = g * voh / (nd > 1e-8f ? nd : 1e-8f);
            const float fc = libm::pow5f(1.f - voh);
            a += (1.f - fc) * gv;
            b += fc * gv;
        }
    }
    out[i] = make_float2(a / (float)n_samples, b / (float)n_samples);
}

// host table -> context workspace `slot` (synchronous: the table is a
// temporary)
int upload(dressi_ctx* ctx, int slot, const std::vector<float4>& v, const float4** out) {
    void* p = nullptr;
    if (int rc = ctx_workspace(ctx, slot, v.size() * sizeof(float4), &p)) return rc;
    DRESSI_TRY_HIP(hipMemcpyAsync(p, v.data(), v.size() * sizeof(float4), hipMemcpyHostToDevice,
                                  ctx->stream));
    DRESSI_TRY_HIP(hipStreamSynchronize(ctx->stream));
    *out = (const float4*)p;
    return DRESSI_OK;
}

enum TableKind : int { kDirs = 0, kSamples = 1 };

// The texel directions of an (a, b) map (kDirs) or the a angles of a sample
// count (kSamples). They depend on the sizes alone, but the C library's sinf
// and cosf per texel, the copy and the wait for it took 40-150 us of host
// time per table and call (28 tables, ~1 ms, in the chain of a 512 x 256
// environment whose kernels take 0.8 ms). So the context keeps them: up to
// kTablesMax tables of kTableBytesMax each and kTablesBytes together, the
// longest unused given back first. A call uses at most two, and two always
// fit, so the second never takes the first's place. Larger ones go through
// the workspace `slot` on each call, as all did.
constexpr size_t kTableBytesMax = 16u << 20;
constexpr size_t kTablesBytes = 64u << 20;
constexpr size_t kTablesMax = 64;

int device_table(dressi_ctx* ctx, int slot, TableKind kind, uint32_t a, uint32_t b,
                 const float4** out) {
    // a graph would keep the table's address past its place here
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    DRESSI_TRY_HIP(hipStreamIsCapturing(ctx->stream, &capture));
    if (capture != hipStreamCaptureStatusNone) {
        set_error("the IBL convolutions and sample tables cannot be captured");
        return DRESSI_ERR_HIP;
    }
    auto& tables = ctx->tables;
    for (dressi_ctx::Table& t : tables) {
        if (t.kind == kind && t.a == a && t.b == b) {
            t.used = ++ctx->table_clock;
            *out = (const float4*)t.ptr;
            return DRESSI_OK;
        }
    }
    const std::vector<float4> v = kind == kDirs ? host_equirect_dirs(a, b) : host_hammersley(a);
    const size_t bytes = v.size() * sizeof(float4);
    if (bytes > kTableBytesMax) {
        return upload(ctx, slot, v, out);
    }
    size_t total = bytes;
    for (const dressi_ctx::Table& t : tables) total += t.bytes;
    while (tables.size() >= kTablesMax || total > kTablesBytes) {
        const auto old = std::min_element(
                tables.begin(), tables.end(),
                [](const dressi_ctx::Table& x, const dressi_ctx::Table& y) {
                    return x.used < y.used;
                });
        // whatever stream last read it
        DRESSI_TRY_HIP(hipDeviceSynchronize());
        DRESSI_TRY_HIP(hipFree(old->ptr));
        total -= old->bytes;
        tables.erase(old);
    }
    void* p = nullptr;
    DRESSI_TRY_HIP(hipMalloc(&p, bytes));
    // complete before the call returns, so that a later call may read it on
    // any stream
    hipError_t e = hipMemcpyAsync(p, v.data(), bytes, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        hipFree(p);
        set_error("table upload failed: %s", hipGetErrorString(e));
        return DRESSI_ERR_HIP;
    }
    tables.push_back({kind, a, b, p, bytes, ++ctx->table_clock});
    *out = (const float4*)p;
    return DRESSI_OK;
}

template <int MODE>
int run_conv(dressi_ctx* ctx, const float* in, uint32_t sw, uint32_t sh, uint32_t n,
             uint32_t ow, uint32_t oh, float alpha, const float* norm, float* out) {
    const float4 *od = nullptr, *sd = nullptr;
    if (int rc = device_table(ctx, 10, kDirs, ow, oh, &od)) return rc;
    if (int rc = device_table(ctx, 11, kDirs, sw, sh, &sd)) return rc;
    constexpr bool kBwd = MODE == kIrrBwd || MODE == kPrefBwd;
    const uint32_t n_i = kBwd ? sw * sh : ow * oh;
    const float scale = kIblTwoPi / ((float)sw * (float)sh);
    const bool few = n_i <= kFewMax;
    const auto launch = [&](auto n_comp) {
        constexpr int N = decltype(n_comp)::value;
        const auto kernel = few ? k_eq_conv_few<MODE, N> : k_eq_conv<MODE, N>;
        const uint32_t per = few ? kFewOut : kConvOut;
        constexpr uint32_t kBlocks = (uint32_t)(kLaunchThreads / kConvThreads);
        for (uint32_t first = 0; first < n_i; first += kBlocks * per) {
            hipLaunchKernelGGL(kernel, dim3(std::min(div_up(n_i - first, per), kBlocks)),
                               dim3(kConvThreads), 0, ctx->stream, od, ow * oh, sd, sw * sh, in,
                               norm, alpha, scale, first, out);
        }
    };
    switch (MODE == kPrefNorm ? 1u : n) {
        case 1: launch(std::integral_constant<int, 1>()); break;
        case 2: launch(std::integral_constant<int, 2>()); break;
        case 3: launch(std::integral_constant<int, 3>()); break;
        default: launch(std::integral_constant<int, 4>()); break;
    }
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int check_map(uint32_t w, uint32_t h, uint32_t n) {
    DRESSI_REQUIRE(n >= 1 && n <= 4, "n_comp must be 1..4");
    DRESSI_REQUIRE(w > 0 && h > 0 && (uint64_t)w * h < (1ull << 28), "bad map size %ux%u", w, h);
    return DRESSI_OK;
}

}  // namespace
}  // namespace dressi

using namespace dressi;

extern "C" {

int dressi_equirect_sample(dressi_ctx* ctx, const float* map, uint32_t mw, uint32_t mh,
                           uint32_t n_comp, const float* dir, uint32_t dw, uint32_t dh,
                           float* out) {
    DRESSI_REQUIRE(ctx && map && dir && out, "bad arguments");
    if (int rc = check_map(mw, mh, n_comp)) return rc;
    const size_t npx = (size_t)dw * dh;
    if (!npx) return DRESSI_OK;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_eq_sample, dim3((uint32_t)((npx + 255) / 256)), dim3(256), 0,
                       ctx->stream, map, (int)mw, (int)mh, n_comp, dir, npx, out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_equirect_sample_bwd(dressi_ctx* ctx, const float* gy, uint32_t n_comp,
                               const float* dir, uint32_t dw, uint32_t dh, uint32_t mw,
                               uint32_t mh, float* out) {
    DRESSI_REQUIRE(ctx && gy && dir && out, "bad arguments");
    if (int rc = check_map(mw, mh, n_comp)) return rc;
    const size_t npx = (size_t)dw * dh, cnt = (size_t)mw * mh * n_comp;
    DRESSI_REQUIRE(npx < (1ull << 40), "too many pixels");
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    void *acc = nullptr, *mx = nullptr;
    if (int rc = ctx_workspace(ctx, 12, cnt * sizeof(unsigned long long), &acc)) return rc;
    if (int rc = ctx_workspace(ctx, 13, kScatterParts * sizeof(uint32_t), &mx)) return rc;
    const size_t ng = npx * n_comp;
    const uint32_t n_part =
            (uint32_t)std::min<size_t>((std::max(ng, cnt) + 1023) / 1024, kScatterParts);
    hipLaunchKernelGGL(k_eq_scatter_prep, dim3(n_part), dim3(256), 0, ctx->stream, gy, ng,
                       (uint32_t*)mx, (unsigned long long*)acc, cnt);
    DRESSI_CHECK_LAUNCH();
    if (npx) {
        // square tiles where the image has the rows and columns for them,
        // flat or narrow ones for a list of directions
        uint32_t tile_h = 1;
        while (tile_h < 32 && tile_h < dh) tile_h *= 2;
        while (tile_h < kScatterPixels && kScatterPixels / tile_h >= 2ull * dw) tile_h *= 2;
        const uint32_t tile_w = kScatterPixels / tile_h;
        const uint32_t tiles_x = div_up(dw, tile_w);
        const uint64_t tiles = (uint64_t)tiles_x * div_up(dh, tile_h);
        DRESSI_REQUIRE(tiles < (1ull << 31), "too many pixels");
        uint32_t copies_log2 = 0, slots_log2 = 0;
        if (cnt <= kScatterDirect) {
            while (copies_log2 < 5 && cnt << (copies_log2 + 1) <= kScatterDirect) copies_log2++;
        } else {
            // four sums per texel in a quarter of the slots where an image
            // that covers the map gives a texel 16 pixels and more; a tile
            // with more texels than slots adds the rest in memory
            copies_log2 = npx / 16 >= (size_t)mw * mh ? kScatterHashCopies : 0u;
            slots_log2 = scatter_slots_log2(n_comp) - copies_log2;
        }
        const size_t sums = slots_log2 ? (size_t)n_comp << slots_log2 : cnt;
        const size_t lds = (sums << copies_log2) * 8 + (slots_log2 ? 4ull << slots_log2 : 0);
        constexpr uint32_t kBlocks = (uint32_t)(kLaunchThreads / kScatterThreads);
        for (uint32_t tile0 = 0; tile0 < (uint32_t)tiles; tile0 += kBlocks) {
            hipLaunchKernelGGL(k_eq_scatter, dim3(std::min((uint32_t)tiles - tile0, kBlocks)),
                               dim3(kScatterThreads), lds, ctx->stream, gy, n_comp, dir, dw, dh,
                               tile_w, tiles_x, (int)mw, (int)mh, (const uint32_t*)mx, n_part,
                               slots_log2, copies_log2, tile0, (unsigned long long*)acc);
            DRESSI_CHECK_LAUNCH();
        }
    }
    hipLaunchKernelGGL(k_fixed_resolve, dim3((uint32_t)((cnt + 255) / 256)), dim3(256), 0,
                       ctx->stream, (const unsigned long long*)acc, cnt, (const uint32_t*)mx,
                       n_part, (double)npx, out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_avg_pool2x2(dressi_ctx* ctx, const float* x, uint32_t w, uint32_t h, uint32_t n_comp,
                       float* out) {
    DRESSI_REQUIRE(ctx && x && out, "bad arguments");
    if (int rc = check_map(w, h, n_comp)) return rc;
    const uint32_t ow = (w + 1) / 2, oh = (h + 1) / 2;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_pool_fwd, dim3(div_up(ow * oh, 256)), dim3(256), 0, ctx->stream, x,
                       (int)w, (int)h, n_comp, (int)ow, (int)oh, out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_avg_pool2x2_bwd(dressi_ctx* ctx, const float* gy, uint32_t w, uint32_t h,
                           uint32_t n_comp, float* out) {
    DRESSI_REQUIRE(ctx && gy && out, "bad arguments");
    if (int rc = check_map(w, h, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_pool_bwd, dim3(div_up(w * h, 256)), dim3(256), 0, ctx->stream, gy,
                       (int)w, (int)h, n_comp, (int)((w + 1) / 2), out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_irradiance_conv(dressi_ctx* ctx, const float* env, uint32_t sw, uint32_t sh,
                           uint32_t n_comp, uint32_t ow, uint32_t oh, float* out) {
    DRESSI_REQUIRE(ctx && env && out, "bad arguments");
    if (int rc = check_map(sw, sh, n_comp)) return rc;
    if (int rc = check_map(ow, oh, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    return run_conv<kIrrFwd>(ctx, env, sw, sh, n_comp, ow, oh, 0.f, nullptr, out);
}

int dressi_irradiance_conv_bwd(dressi_ctx* ctx, const float* gy, uint32_t ow, uint32_t oh,
                               uint32_t n_comp, uint32_t sw, uint32_t sh, float* out) {
    DRESSI_REQUIRE(ctx && gy && out, "bad arguments");
    if (int rc = check_map(sw, sh, n_comp)) return rc;
    if (int rc = check_map(ow, oh, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    return run_conv<kIrrBwd>(ctx, gy, sw, sh, n_comp, ow, oh, 0.f, nullptr, out);
}

int dressi_prefilter_conv_norm(dressi_ctx* ctx, uint32_t ow, uint32_t oh, uint32_t sw,
                               uint32_t sh, float roughness, float* out) {
    DRESSI_REQUIRE(ctx && out, "bad arguments");
    if (int rc = check_map(sw, sh, 1)) return rc;
    if (int rc = check_map(ow, oh, 1)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    const float r = roughness > 0.045f ? roughness : 0.045f;
    return run_conv<kPrefNorm>(ctx, nullptr, sw, sh, 1, ow, oh, r * r, nullptr, out);
}

int dressi_prefilter_conv(dressi_ctx* ctx, const float* env, uint32_t sw, uint32_t sh,
                          uint32_t n_comp, uint32_t ow, uint32_t oh, float roughness,
                          const float* norm, float* out) {
    DRESSI_REQUIRE(ctx && env && norm && out, "bad arguments");
    if (int rc = check_map(sw, sh, n_comp)) return rc;
    if (int rc = check_map(ow, oh, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    const float r = roughness > 0.045f ? roughness : 0.045f;
    return run_conv<kPrefFwd>(ctx, env, sw, sh, n_comp, ow, oh, r * r, norm, out);
}

int dressi_prefilter_conv_bwd(dressi_ctx* ctx, const float* gy, uint32_t ow, uint32_t oh,
                              uint32_t n_comp, uint32_t sw, uint32_t sh, float roughness,
                              const float* norm, float* out) {
    DRESSI_REQUIRE(ctx && gy && norm && out, "bad arguments");
    if (int rc = check_map(sw, sh, n_comp)) return rc;
    if (int rc = check_map(ow, oh, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    const float r = roughness > 0.045f ? roughness : 0.045f;
    return run_conv<kPrefBwd>(ctx, gy, sw, sh, n_comp, ow, oh, r * r, norm, out);
}

int dressi_prefilter_env(dressi_ctx* ctx, const float* env, uint32_t sw, uint32_t sh,
                         uint32_t n_comp, uint32_t ow, uint32_t oh, float roughness,
                         uint32_t n_samples, float* out) {
    DRESSI_REQUIRE(ctx && env && out, "bad arguments");
    DRESSI_REQUIRE(n_samples > 0, "n_samples must be > 0");
    if (int rc = check_map(sw, sh, n_comp)) return rc;
    if (int rc = check_map(ow, oh, n_comp)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    const float4 *od = nullptr, *smp = nullptr;
    if (int rc = device_table(ctx, 10, kDirs, ow, oh, &od)) return rc;
    if (int rc = device_table(ctx, 11, kSamples, n_samples, 0, &smp)) return rc;
    hipLaunchKernelGGL(k_prefilter_env, dim3(div_up(ow * oh, 64)), dim3(64), 0, ctx->stream, od,
                       ow * oh, env, (int)sw, (int)sh, n_comp, smp, n_samples, roughness, out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

int dressi_brdf_lut(dressi_ctx* ctx, uint32_t w, uint32_t h, uint32_t n_samples, float* out) {
    DRESSI_REQUIRE(ctx && out, "bad arguments");
    DRESSI_REQUIRE(n_samples > 0, "n_samples must be > 0");
    if (int rc = check_map(w, h, 2)) return rc;
    DRESSI_TRY_HIP(hipSetDevice(ctx->device));
    const float4* smp = nullptr;
    if (int rc = device_table(ctx, 11, kSamples, n_samples, 0, &smp)) return rc;
    hipLaunchKernelGGL(k_brdf_lut, dim3(div_up(w * h, 64)), dim3(64), 0, ctx->stream, (int)w,
                       (int)h, smp, n_samples, (float2*)out);
    DRESSI_CHECK_LAUNCH();
    return DRESSI_OK;
}

}  // extern "C"
