// raster.hip -- shadow-map depth pass and the camera G-buffer (depth pre-pass
// + per-pixel surface attributes) on the binned rasterizer.
//
// Shadow map: simple.vert draws every actor with projection*view of the light
// (src/Application.cpp:212-233); only depth matters for cone tracing.
// G-buffer: the depth pre-pass (src/Application.cpp:936-965) plus what
// phong.vert hands phong.frag (shaders/phong.vert:36-59): world position,
// normal, and the TBN columns.  Visibility is an order-independent 64-bit
// atomicMin of (depth bits, ~triangle id): the nearest fragment wins and, at
// equal depth, the triangle drawn last wins, as glDepthFunc(GL_EQUAL) shading
// after the pre-pass does.
#pragma clang fp contract(off)

#include <algorithm>

#include "raster_common.h"
#include "texture.h"

namespace vctk {

__device__ __forceinline__ void world_vertex(const DevScene &sc, int t, int v, float w[3]) {
    const float *M = sc.model + (size_t)sc.obj[t] * 16;
    const float *p = sc.pos + (size_t)t * 9 + v * 3;
    float p4[4] = {p[0], p[1], p[2], 1.0f}, o[4];
    mat4_vec4(M, p4, o);
    w[0] = o[0];
    w[1] = o[1];
    w[2] = o[2];
}

// ---------------------------------------------------------------- shadow map
// One walk draws up to kShadowBatch lights' maps: slot j * ntri + t is
// triangle t seen from the walk's j-th light, whose index in the light array
// sits at bits 5j .. 5j+4 of `li` (light indices are below kMaxLights = 32).
// Each map receives exactly the fragments a walk of its light alone gives it
// (depth is an order-independent atomicMin), so the batching does not change
// a texel.
static_assert(kMaxLights <= 32, "light indices are packed in 5 bits");
static_assert(kShadowBatch * 5 <= 64, "a walk's light indices fit one 64-bit argument");

// A triangle whose bounding box holds more than this many pixels is drawn by
// the block walk (k_raster_blocks), the others by the pixel walk.
constexpr uint64_t kBlockPixels = 256;

// The 8x8 pixel blocks (aligned to multiples of 8) that cover the bounding box
// of a setup record r with cnt bounding-box pixels.
__device__ __forceinline__ uint64_t bbox_blocks(const int4 r[4], uint64_t cnt) {
    const int x0 = r[1].z & 0xffff, y0 = (int)((uint32_t)r[1].z >> 16), bw = r[1].w & 0xffff;
    const int bh = (int)(cnt / (uint64_t)bw);
    const uint64_t nbx = (uint64_t)(((x0 + bw - 1) >> 3) - (x0 >> 3) + 1);
    const uint64_t nby = (uint64_t)(((y0 + bh - 1) >> 3) - (y0 >> 3) + 1);
    return nbx * nby;
}

// A record for the block walk, whose FP64 sums start from the edge values C at the
// origin, every sum exact.  |A|, |B| <= 2^28 and a pixel centre is below 2^22 in
// 1/256 px, an odd multiple of 128: the terms in A and B are multiples of 128 and
// together at most 2^51.  With C below 2^52 every sum is an integer below 2^53.  From
// there on (C is at most 2^55) the edge passes far from the image: no sum changes its
// sign, and the values lie between 2^51 and 2^56, where floats and the midpoints
// between them are multiples of 2^27.  So all values from one multiple of 128 to the
// next, ends excluded, round to the same float, and C's remainder mod 128 may be 64
// wherever it is not 0: multiples of 64 below 2^56 are exact again.
__device__ __forceinline__ void walk_record(int4 r[4]) {
    if (((uint32_t)r[1].w >> 19) & 1u) return;  // small: 32-bit values
    int *const w[3][2] = {{&r[2].x, &r[2].y}, {&r[2].z, &r[2].w}, {&r[3].x, &r[3].y}};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t c = (int64_t)(((uint64_t)(uint32_t)*w[i][1] << 32) | (uint32_t)*w[i][0]);
        const bool far = (uint64_t)(c + ((int64_t)1 << 52)) >= ((uint64_t)1 << 53);
        if (far) *w[i][0] = (*w[i][0] & ~127) | ((*w[i][0] & 127) ? 64 : 0);
    }
}

// Words of `w` to v, by `threads` threads of which this is the t-th: 16 bytes
// at a time (w is the start of an allocation).
__device__ __forceinline__ void fill_words(uint32_t *w, uint32_t v, size_t n, size_t t, size_t threads) {
    for (size_t i = t; i < n / 4; i += threads) ((uint4 *)w)[i] = make_uint4(v, v, v, v);
    if (t < (n & 3)) w[(n & ~(size_t)3) + t] = v;
}

// Workgroups of a set-up kernel that also clears `words` words of an image: its
// triangles', and no fewer than the clear fills (4 stores a thread, up to 4
// workgroups per CU).  The clear's writes run beside the set-up's own work: five
// 1024^2 maps took 5 launches of 5.7 us before, now 4 us of the set-up's.
inline unsigned setup_blocks(int ntri, size_t words) {
    const size_t tri = ((size_t)ntri + 255) / 256, fill = (words + 4095) / 4096;
    return (unsigned)std::max(tri, std::min(fill, (size_t)1024));
}

__global__ __launch_bounds__(256) void k_shadow_setup(DevScene sc, const DevLight *__restrict__ lights, uint64_t li,
                                                      int4 *rec, float4 *attr, uint32_t *counts, uint32_t *bcounts) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int l = (int)((li >> (5u * blockIdx.y)) & 31u);
    const float *ls = lights[l].ls;
    const int N = (int)lights[l].shadow_size;
    fill_words((uint32_t *)const_cast<float *>(lights[l].shadowmap), 0x3f800000u, (size_t)N * N, t,
               gridDim.x * blockDim.x);  // clear depth 1.0
    if (t >= sc.ntri) return;
    const size_t slot = (size_t)blockIdx.y * (size_t)sc.ntri + (size_t)t;
    float clip[3][4];
    bool behind = false;
    for (int v = 0; v < 3; ++v) {
        float w[3];
        world_vertex(sc, t, v, w);
        float w4[4] = {w[0], w[1], w[2], 1.0f};
        mat4_vec4(ls, w4, clip[v]);
        if (clip[v][2] < -clip[v][3] || clip[v][3] <= 0.0f) behind = true;
    }
    uint64_t cnt = 0;
    if (!behind) {
        float half = (float)N * 0.5f;
        float win[3][2], zw[3];
        for (int v = 0; v < 3; ++v) {
            float xd = clip[v][0] / clip[v][3], yd = clip[v][1] / clip[v][3], zd = clip[v][2] / clip[v][3];
            win[v][0] = xd * half + half;
            win[v][1] = yd * half + half;
            zw[v] = zd * 0.5f + 0.5f;
        }
        int4 r[4];
        // back faces culled: GL_CULL_FACE stays enabled from the previous
        // frame's passes when the reference draws its shadow map
        // (Application.cpp:737,942,979); the record's user field is the light
        cnt = tri_setup(win, N, N, 1, l, r);
        if (cnt) {
            if (cnt > kBlockPixels) walk_record(r);
            for (int i = 0; i < 4; ++i) rec[slot * 4 + i] = r[i];
            attr[slot] = make_float4(zw[0], zw[1], zw[2], 0.0f);
        }
        if (cnt > kBlockPixels) {  // 8x8 blocks of the bounding box instead of its pixels
            counts[slot] = 0;
            bcounts[slot] = (uint32_t)bbox_blocks(r, cnt);
            return;
        }
    }
    counts[slot] = (uint32_t)cnt;
    bcounts[slot] = 0;
}

// The large triangles of a walk, 8x8-pixel blocks of their bounding boxes, the
// lanes a block's pixels (row-major).  A wavefront takes runs of consecutive
// blocks (up to kBlockRun; run r by wavefront r % wavefronts, so that the runs
// of covered blocks and of empty ones are dealt out evenly), and a triangle's
// record is wave-uniform: its slot is found in the offsets of up to 64 slots that
// the lanes hold, read where a run begins or passes their end.  (A table of every
// block's slot, filled by a launch of its own, took 10 to 23 us and left the walk
// no faster: 534 us with it, 507 without.)  Each lane keeps its three edge values
// in FP64 and steps them from block to block, every sum exact (walk_record), so the
// values round to float as those of edge_value do in both of its forms, and the
// barycentrics are quot_f32(E, area) with the triangle's reciprocal: every fragment
// and its barycentrics are those the pixel walk produces.  F provides Tri (a triangle's
// wave-uniform data, the image size W x H among it), enter(slot, edges) that
// gives it, and three stages of a fragment, between which a Pending goes:
// fetch(tri, px, py, in), depth(tri, l, pending) and store(pending), which runs
// after the wavefront's next covered block has been fetched.
//
// What bounds it: VALU issue and the scalar work beside it (an empty block 3
// additions and 3 comparisons, a covered one 12 more for the quotients and 8
// for the depth), then the atomics, which a load of the word before them spares
// where a nearer fragment is already there.  It was 20 and 45 vector
// instructions a block, in two forms (32-bit and FP64) whose arrays took 82
// registers: 5 wavefronts per SIMD for a grid of 8, on equal shares of
// consecutive blocks.  Five 1024^2 maps: 286 us before, 183; five 2048^2 maps:
// 1024 us before, 507.  The load in the same stage as the atomic suits the depth
// maps (190 and 560 us with the G-buffer's stages); the G-buffer, fewer blocks
// of longer triangles, waits for the load, so the atomic goes one block later
// (1920x1080: 79 us without the load, 92 with it, 73 one block later; 3840x2160:
// 427, 271, 254).

constexpr int kBlockRun = 64;

template <class F>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_raster_blocks(
    const int4 *__restrict__ recs, const uint64_t *__restrict__ offs, const uint32_t *__restrict__ chunk,
    size_t chunk_cap, int nslots, F f) {
    const uint64_t total = offs[nslots];
    const uint64_t nchunks = (total + 63) >> 6;
    const int lane = threadIdx.x & 63;
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const uint64_t share = (total + nwaves - 1) / nwaves;
    const uint64_t run = share < (uint64_t)kBlockRun ? (share ? share : 1) : (uint64_t)kBlockRun;
    typename F::Pending last = {};
    const double dxl = (double)((lane & 7) * 256 + 128), dyl = (double)((lane >> 3) * 256 + 128);
    for (uint64_t r0 = wave * run; r0 < total; r0 += nwaves * run) {
        const uint64_t r1 = r0 + run < total ? r0 + run : total;
        uint64_t k = r0;
        int lo = 0, known = 0;       // lane i holds the offset of slot lo + i, for `known` slots
        uint64_t off = 0;
        while (k < r1) {  // the run's next triangle
            uint64_t m = __ballot(lane < known && off <= k);
            if (m == 0 || m >> (known - 1) != 0) {  // not among the slots at hand
                const uint64_t c = k >> 6;          // block k lies in chunk c (64 blocks per chunk)
                const int first = c < chunk_cap ? (int)chunk[c] : 0;
                int hi = (c + 1 < nchunks && c + 1 < chunk_cap) ? (int)chunk[c + 1] : nslots - 1;
                lo = __builtin_amdgcn_readfirstlane(lo + known > first && known ? lo + known - 1 : first);
                hi = __builtin_amdgcn_readfirstlane(hi);
                while (hi - lo >= 63) {  // the last slot of [lo, hi] that starts at or before k, 64 probes at a time
                    const int step = ((hi - lo) >> 6) + 1;
                    const int p = lo + lane * step;
                    const int top = 63 - __builtin_clzll(__ballot(p <= hi && offs[p <= hi ? p : hi] <= k));
                    lo += top * step;
                    hi = lo + step - 1 < hi ? lo + step - 1 : hi;
                }
                known = nslots - lo < 63 ? nslots - lo + 1 : 64;
                off = offs[lo + (lane < known ? lane : 0)];
                m = __ballot(lane < known && off <= k);
            }
            const int at = 63 - __builtin_clzll(m);
            const int slot = lo + at;
            const uint64_t t0 = readlane_u64(off, at), t1 = readlane_u64(off, at + 1);
            const uint32_t n = (uint32_t)((t1 < r1 ? t1 : r1) - k);  // its blocks in this run
            Edges e;
            load_edges(recs, (size_t)slot, e);
            const typename F::Tri tri = f.enter(slot, e);
            const uint32_t nbx = (uint32_t)(((e.x0 + e.bw - 1) >> 3) - (e.x0 >> 3) + 1);
            const uint32_t local = (uint32_t)(k - t0);  // the run may enter a triangle mid-way
            uint32_t bxi = __builtin_amdgcn_readfirstlane(local % nbx);
            const int bx0 = (e.x0 >> 3) * 8, by = ((e.y0 >> 3) + (int)(local / nbx)) * 8;
            const double rcp = rcp_f64(e.area);
            double E[3], row[3], As[3], Bs[3], lim[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double A = (double)e.A[i], B = (double)e.B[i];
                // the small form's edge value at the bounding box corner, as the
                // value at the origin
                const double C = e.small ? (double)e.E0[i] - (A * (double)(e.x0 << 8) + B * (double)(e.y0 << 8))
                                         : (double)e.C[i];
                row[i] = fma(A, (double)(bx0 * 256) + dxl, fma(B, (double)(by * 256) + dyl, C));
                As[i] = A * 2048.0;
                Bs[i] = B * 2048.0;
                E[i] = fma((double)(int)bxi, As[i], row[i]);
                lim[i] = (double)(-e.bias[i]);
            }
            int px = bx0 + (int)bxi * 8 + (lane & 7), py = by + (lane >> 3);
            for (uint32_t j = 0; j < n; ++j) {
                // px, py: outside where the block overhangs the image
                const bool in = (E[0] >= lim[0]) & (E[1] >= lim[1]) & (E[2] >= lim[2]) & (px < tri.W) & (py < tri.H);
                if (__ballot(in) != 0) {  // an empty block ends here
                    typename F::Pending cur = f.fetch(tri, px, py, in);
                    float l[3];
#pragma unroll
                    for (int i = 0; i < 3; ++i) l[i] = quot_f32((float)E[i], rcp);
                    f.depth(tri, l, cur);
                    f.store(last);  // the last covered block's: its word has arrived by now
                    last = cur;
                }
                if (++bxi == nbx) {
                    bxi = 0;
                    px = bx0 + (lane & 7);
                    py += 8;
#pragma unroll
                    for (int i = 0; i < 3; ++i) E[i] = row[i] = row[i] + Bs[i];
                } else {
                    px += 8;
#pragma unroll
                    for (int i = 0; i < 3; ++i) E[i] = E[i] + As[i];
                }
            }
            k += n;
        }
    }
    f.store(last);
}

// A walk's shadow maps by light index (Edges::user), in the kernel arguments.
struct ShadowMaps {
    uint32_t *map[kMaxLights];
    int size[kMaxLights];
};
typedef __attribute__((address_space(1))) uint32_t global_u32;

// ShadowFrag for the block walk: load, comparison and atomic in one stage.
struct ShadowBlockFrag {
    const float4 *attr;
    ShadowMaps maps;
    struct Tri {
        float4 a;
        global_u32 *map;
        int W, H;
    };
    struct Pending {
        global_u32 *d;
        bool live;
    };
    __device__ Tri enter(int slot, const Edges &e) const {
        Tri t;
        t.a = attr[slot];
        t.map = (global_u32 *)maps.map[e.user];
        t.W = t.H = maps.size[e.user];
        return t;
    }
    __device__ Pending fetch(const Tri &t, int px, int py, bool in) const {
        return Pending{t.map + (uint32_t)(py * t.W + px), in};
    }
    __device__ void depth(const Tri &t, const float l[3], Pending &p) const {
        float z = interp3(l, t.a.x, t.a.y, t.a.z);
        z = z + 0.0f;
        if (p.live && z >= 0.0f && z <= 1.0f) {
            const uint32_t zu = __float_as_uint(z);
            if (__hip_atomic_load(p.d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > zu)  // seen()
                __hip_atomic_fetch_min(p.d, zu, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __device__ void store(const Pending &) const {}
};

struct ShadowFrag {
    const float4 *attr;
    const DevLight *lights;
    __device__ void item(int slot, int px, int py, const Edges &e) {
        if (!edge_inside(e, px, py, 128, 128)) return;
        float l[3];
        edge_bary(e, px, py, 128, 128, l);
        float4 a = attr[slot];
        float z = interp3(l, a.x, a.y, a.z);
        z = z + 0.0f;
        if (!(z >= 0.0f && z <= 1.0f)) return;
        const DevLight &L = lights[e.user];
        uint32_t *depth = (uint32_t *)const_cast<float *>(L.shadowmap);
        atomicMin(&depth[(size_t)py * L.shadow_size + px], __float_as_uint(z));
    }
    __device__ void finish() {}
};

__global__ void k_shadow_pad_batch(const DevLight *__restrict__ lights, uint64_t li);

hipError_t launch_shadowmaps(const DevScene &sc, const DevLight *hlights, const DevLight *dlights, const int *li,
                             int n, RasterScratch &rs, hipStream_t s) {
    hipError_t e;
    const int batch = shadow_batch(sc.ntri);
    for (int j0 = 0; j0 < n; j0 += batch) {
        const int nb = n - j0 < batch ? n - j0 : batch;
        uint64_t packed = 0;
        size_t texels = 0;
        for (int j = 0; j < nb; ++j) {
            const size_t N = hlights[li[j0 + j]].shadow_size;
            if (N * N > texels) texels = N * N;
            packed |= (uint64_t)(uint32_t)li[j0 + j] << (5 * j);
        }
        const size_t nslots = (size_t)nb * (size_t)sc.ntri;
        hipLaunchKernelGGL(k_shadow_setup, dim3(setup_blocks(sc.ntri, texels), nb), dim3(256), 0, s, sc, dlights,
                           packed, rs.rec, rs.attr, rs.counts, rs.bcounts);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (sc.ntri > 0) {
            if ((e = raster_scan(rs, nslots, true, s)) != hipSuccess) return e;
            ShadowFrag f{rs.attr, dlights};
            hipLaunchKernelGGL(k_raster_items<ShadowFrag>, dim3(raster_grid<ShadowFrag, false>()), dim3(256), 0, s,
                               rs.rec, rs.offs, rs.chunk, rs.chunk_cap, (int)nslots, f);
            if ((e = hipGetLastError()) != hipSuccess) return e;
            ShadowBlockFrag fb{};
            fb.attr = rs.attr;
            for (int j = 0; j < nb; ++j) {
                const DevLight &L = hlights[li[j0 + j]];
                fb.maps.map[li[j0 + j]] = (uint32_t *)const_cast<float *>(L.shadowmap);
                fb.maps.size[li[j0 + j]] = (int)L.shadow_size;
            }
            hipLaunchKernelGGL(k_raster_blocks<ShadowBlockFrag>, dim3(kRasterBlocks), dim3(256), 0, s, rs.rec,
                               rs.boffs, rs.bchunk, rs.chunk_cap, (int)nslots, fb);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        // the padded copy of every map of the walk, one launch
        int pmax = 0;
        for (int j = 0; j < nb; ++j) {
            const DevLight &L = hlights[li[j0 + j]];
            if (L.shadowpad) pmax = std::max(pmax, (int)L.shadow_size + 2 * kShadowPad);
        }
        if (pmax > 0) {
            hipLaunchKernelGGL(k_shadow_pad_batch, dim3(pmax, nb), dim3(256), 0, s, dlights, packed);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

// Row blockIdx.x of a padded copy.
__device__ __forceinline__ void shadow_pad_row(const float *__restrict__ sm, int N, float *pad) {
    const int n = N + 2 * kShadowPad, j = (int)blockIdx.x - kShadowPad;
    if ((int)blockIdx.x >= n) return;
    for (int x = threadIdx.x; x < n; x += 256) {
        const int i = x - kShadowPad;
        pad[(size_t)blockIdx.x * n + x] = (i >= 0 && i < N && j >= 0 && j < N) ? sm[(size_t)j * N + i] : 1.0f;
    }
}

__global__ __launch_bounds__(256) void k_shadow_pad(const float *__restrict__ sm, int N, float *pad) {
    shadow_pad_row(sm, N, pad);
}

// The padded copies of a shadow walk's maps: blockIdx.y is the walk's j-th
// light (its index at bits 5j .. 5j+4 of li); lights without a buffer for it
// are skipped.
__global__ __launch_bounds__(256) void k_shadow_pad_batch(const DevLight *__restrict__ lights, uint64_t li) {
    const DevLight &L = lights[(li >> (5u * blockIdx.y)) & 31u];
    if (L.shadowpad) shadow_pad_row(L.shadowmap, (int)L.shadow_size, const_cast<float *>(L.shadowpad));
}

hipError_t launch_shadow_pad(const float *depth, int N, float *pad, hipStream_t s) {
    if (!pad) return hipSuccess;
    hipLaunchKernelGGL(k_shadow_pad, dim3(N + 2 * kShadowPad), dim3(256), 0, s, depth, N, pad);
    return hipGetLastError();
}

// ---------------------------------------------------------------- G-buffer
struct CamMats {
    float pv[16];
    int W, H, cull;
};

__global__ __launch_bounds__(256) void k_gbuf_setup(DevScene sc, CamMats cm, int4 *rec, float4 *attr,
                                                    uint32_t *counts, uint32_t *bcounts, uint32_t *vis) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    fill_words(vis, ~0u, (size_t)cm.W * cm.H * 2, t, gridDim.x * blockDim.x);
    if (t >= sc.ntri) return;
    float clip[3][4];
    for (int v = 0; v < 3; ++v) {
        float w[3];
        world_vertex(sc, t, v, w);
        float w4[4] = {w[0], w[1], w[2], 1.0f};
        mat4_vec4(cm.pv, w4, clip[v]);
    }
    // Sutherland-Hodgman against the near plane z >= -w
    float poly[4][4];
    int n = 0;
    float d[3];
    for (int i = 0; i < 3; ++i) d[i] = clip[i][2] + clip[i][3];
    for (int i = 0; i < 3; ++i) {
        int j = (i + 1) % 3;
        bool ii = d[i] >= 0.0f, jj = d[j] >= 0.0f;
        if (ii) {
            for (int k = 0; k < 4; ++k) poly[n][k] = clip[i][k];
            n++;
        }
        if (ii != jj) {
            float tt = d[i] / (d[i] - d[j]);
            for (int k = 0; k < 4; ++k) poly[n][k] = clip[i][k] + tt * (clip[j][k] - clip[i][k]);
            n++;
        }
    }
    const float hw = (float)cm.W * 0.5f, hh = (float)cm.H * 0.5f;
    for (int sub = 0; sub < 2; ++sub) {
        const size_t slot = (size_t)t * 2 + sub;
        uint64_t cnt = 0;
        if (sub + 2 < n) {  // fan (0,1,2) needs 3 vertices, (0,2,3) needs 4
            const int vi[3] = {0, sub + 1, sub + 2};
            float win[3][2], zw[3];
            bool bad = false;
            for (int v = 0; v < 3; ++v) {
                const float *c = poly[vi[v]];
                float w = c[3];
                if (!(w > 0.0f)) bad = true;
                float xd = c[0] / w, yd = c[1] / w, zd = c[2] / w;
                win[v][0] = xd * hw + hw;
                win[v][1] = yd * hh + hh;
                zw[v] = zd * 0.5f + 0.5f;
            }
            if (!bad) {
                int4 r[4];
                cnt = tri_setup(win, cm.W, cm.H, cm.cull, t, r);
                if (cnt) {
                    if (cnt > kBlockPixels) walk_record(r);
                    for (int i = 0; i < 4; ++i) rec[slot * 4 + i] = r[i];
                    attr[slot] = make_float4(zw[0], zw[1], zw[2], 0.0f);
                }
                if (cnt > kBlockPixels) {  // 8x8 blocks of the bounding box instead of its pixels
                    counts[slot] = 0;
                    bcounts[slot] = (uint32_t)bbox_blocks(r, cnt);
                    continue;
                }
            }
        }
        counts[slot] = (uint32_t)cnt;
        bcounts[slot] = 0;
    }
}

struct GbufFrag {
    const float4 *attr;
    unsigned long long *vis;
    int W;
    __device__ void item(int slot, int px, int py, const Edges &e) {
        if (!edge_inside(e, px, py, 128, 128)) return;
        float l[3];
        edge_bary(e, px, py, 128, 128, l);
        float4 a = attr[slot];
        float z = interp3(l, a.x, a.y, a.z);
        z = z + 0.0f;
        if (!(z >= 0.0f && z <= 1.0f)) return;
        const uint32_t tri = (uint32_t)e.user;
        unsigned long long key = ((unsigned long long)__float_as_uint(z) << 32) | (unsigned long long)(0xffffffffu - tri);
        atomicMin(&vis[(size_t)py * W + px], key);
    }
    __device__ void finish() {}
};

// GbufFrag for the block walk.
struct GbufBlockFrag {
    const float4 *attr;
    unsigned long long *vis;
    int W, H;
    struct Tri {
        float4 a;
        uint32_t low;  // the key's low word: ~triangle
        int W, H;
    };
    struct Pending {
        unsigned long long key, seen;
        uint32_t at;
        bool live;
    };
    __device__ Tri enter(int slot, const Edges &e) const { return Tri{attr[slot], 0xffffffffu - (uint32_t)e.user, W, H}; }
    __device__ Pending fetch(const Tri &, int px, int py, bool in) const {
        Pending p;
        p.at = (uint32_t)(py * W + px);
        p.key = p.seen = 0ull;
        p.live = in;
        if (in) p.seen = vctk::seen(&vis[p.at]);
        return p;
    }
    __device__ void depth(const Tri &t, const float l[3], Pending &p) const {
        float z = interp3(l, t.a.x, t.a.y, t.a.z);
        z = z + 0.0f;
        p.live = p.live && z >= 0.0f && z <= 1.0f;
        p.key = ((unsigned long long)__float_as_uint(z) << 32) | (unsigned long long)t.low;
    }
    __device__ void store(const Pending &p) const {
        if (p.live && p.seen > p.key) atomicMin(&vis[p.at], p.key);
    }
};

// The attributes of the visible triangle at pixel (px, py), as the texel's four
// float4.
__device__ __forceinline__ void resolve_pixel(const DevScene &sc, const CamMats &cm, unsigned long long key, int px,
                                              int py, float4 o[4]) {
    const int t = (int)(0xffffffffu - (uint32_t)(key & 0xffffffffull));
    const float xn = (2.0f * ((float)px + 0.5f)) / (float)cm.W - 1.0f;
    const float yn = (2.0f * ((float)py + 0.5f)) / (float)cm.H - 1.0f;
    float Wp[3][3], clip[3][4];
    for (int v = 0; v < 3; ++v) {
        world_vertex(sc, t, v, Wp[v]);
        float w4[4] = {Wp[v][0], Wp[v][1], Wp[v][2], 1.0f};
        mat4_vec4(cm.pv, w4, clip[v]);
    }
    float ax[3], ay[3];
    for (int v = 0; v < 3; ++v) {
        ax[v] = clip[v][0] - xn * clip[v][3];
        ay[v] = clip[v][1] - yn * clip[v][3];
    }
    float b[3];
    b[0] = ax[1] * ay[2] - ay[1] * ax[2];
    b[1] = ax[2] * ay[0] - ay[2] * ax[0];
    b[2] = ax[0] * ay[1] - ay[0] * ax[1];
    const float sum = (b[0] + b[1]) + b[2];
    const double rsum = rcp_f64(sum);  // the three IEEE quotients b[v] / sum (quot_f32)
    for (int v = 0; v < 3; ++v) b[v] = quot_f32(b[v], rsum);
    const float *Nm = sc.nmat + (size_t)sc.obj[t] * 9;
    float Tw[3];
    mat3_vec3(Nm, sc.tan + (size_t)t * 3, Tw);
    float Nv[3][3], Tv[3][3], Bv[3][3];
    for (int v = 0; v < 3; ++v) {
        mat3_vec3(Nm, sc.nrm + (size_t)t * 9 + v * 3, Nv[v]);
        // phong.vert:48-52 per vertex: T = normalMatrix * tangent, re-orthogonalized against N
        if (sc.vtan) mat3_vec3(Nm, sc.vtan + (size_t)t * 9 + v * 3, Tw);
        float dtn = dot3(Tw, Nv[v]);
        float tt[3] = {Tw[0] - dtn * Nv[v][0], Tw[1] - dtn * Nv[v][1], Tw[2] - dtn * Nv[v][2]};
        nrm3(tt, Tv[v]);
        cross3(Nv[v], Tv[v], Bv[v]);
    }
    float P[3], N[3], T[3], B[3];
    for (int k = 0; k < 3; ++k) {
        P[k] = interp3(b, Wp[0][k], Wp[1][k], Wp[2][k]);
        N[k] = interp3(b, Nv[0][k], Nv[1][k], Nv[2][k]);
        T[k] = interp3(b, Tv[0][k], Tv[1][k], Tv[2][k]);
        B[k] = interp3(b, Bv[0][k], Bv[1][k], Bv[2][k]);
    }
    uint32_t alb = sc.albedo[t];
    const int tid = sc.texid ? sc.texid[t] : -1;
    if (tid >= 0) {  // texture(diffuseMap, fragTexcoord) (phong.frag:449), stored as RGBA8
        const float *st = sc.uv + (size_t)t * 6;
        const float ts = interp3(b, st[0], st[2], st[4]), tt = interp3(b, st[1], st[3], st[5]);
        float rho2 = 0.0f;
        if (tid < sc.tex.count) {
            // The unnormalized barycentrics (before the division by sum) are
            // affine in NDC: d/dxn of b[i] is cy_j cw_k - cw_j cy_k and d/dyn
            // is cw_j cx_k - cx_j cw_k, (i, j, k) cyclic, so ds/dxn =
            // sum_i d b[i]/dxn (s_i - s) / sum exactly; one pixel is 2/W (2/H) in NDC.
            float gx[3], gy[3];
            for (int i = 0; i < 3; ++i) {
                const int j = (i + 1) % 3, k = (i + 2) % 3;
                gx[i] = clip[j][1] * clip[k][3] - clip[j][3] * clip[k][1];
                gy[i] = clip[j][3] * clip[k][0] - clip[j][0] * clip[k][3];
            }
            const int4 inf = sc.tex.info[tid];
            const float TW = (float)inf.y, TH = (float)inf.z;
            const float kx = 2.0f / (float)cm.W, ky = 2.0f / (float)cm.H;
            const float sx = (gx[0] * (st[0] - ts) + gx[1] * (st[2] - ts)) + gx[2] * (st[4] - ts);
            const float tx = (gx[0] * (st[1] - tt) + gx[1] * (st[3] - tt)) + gx[2] * (st[5] - tt);
            const float sy = (gy[0] * (st[0] - ts) + gy[1] * (st[2] - ts)) + gy[2] * (st[4] - ts);
            const float ty = (gy[0] * (st[1] - tt) + gy[1] * (st[3] - tt)) + gy[2] * (st[5] - tt);
            const float dudx = ((sx / sum) * kx) * TW, dvdx = ((tx / sum) * kx) * TH;
            const float dudy = ((sy / sum) * ky) * TW, dvdy = ((ty / sum) * ky) * TH;
            rho2 = fmaxf(dudx * dudx + dvdx * dvdx, dudy * dudy + dvdy * dvdy);
        }
        const float4 c = tex_sample(sc.tex, tid, ts, tt, rho2);
        alb = pack_unorm4x8(c.x, c.y, c.z, c.w);
    }
    const float rough = sc.rough ? sc.rough[sc.obj[t]] : 0.5f;
    o[0] = make_float4(P[0], P[1], P[2], __uint_as_float(alb));
    o[1] = make_float4(N[0], N[1], N[2], rough);
    o[2] = make_float4(T[0], T[1], T[2], __uint_as_float(1u));
    o[3] = make_float4(B[0], B[1], B[2], __uint_as_float((uint32_t)t));
}

// One pixel per lane, 16x16 per workgroup.  What bounds it: the 64 bytes written
// per pixel.  A lane's own four stores go to 32 lines each, so the texels change
// places through LDS and a wavefront stores its four rows of 16 pixels, 1 KB
// each: 1280x720 26.8 us before, 18.3; 1920x1080 56.7, 37; 3840x2160 231, 164
// (a tile of 64x4, 4 KB per row, the same).  The LDS slots of a pixel are rotated
// so that neither side of the exchange has bank conflicts.
__global__ __launch_bounds__(256) void k_gbuf_resolve(DevScene sc, CamMats cm, const unsigned long long *vis,
                                                      vct_gbuffer_texel *out) {
    __shared__ float4 lds[4][256];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int px = blockIdx.x * 16 + (lane & 15), py0 = blockIdx.y * 16 + w * 4, py = py0 + (lane >> 4);
    float4 o[4];
    o[0] = o[1] = o[2] = o[3] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (px < cm.W && py < cm.H) {
        const unsigned long long key = vis[(size_t)py * cm.W + px];
        if (key != ~0ull) resolve_pixel(sc, cm, key, px, py, o);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) lds[w][lane * 4 + ((k + (lane >> 1)) & 3)] = o[k];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int x = blockIdx.x * 16 + (lane >> 2);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int p = r * 16 + (lane >> 2);
        if (x < cm.W && py0 + r < cm.H)
            ((float4 *)&out[(size_t)(py0 + r) * cm.W + x])[lane & 3] = lds[w][p * 4 + (((lane & 3) + (p >> 1)) & 3)];
    }
}

hipError_t launch_gbuffer(const DevScene &sc, const vct_camera &cam, uint64_t *vis, vct_gbuffer_texel *gbuf,
                          RasterScratch &rs, hipStream_t s) {
    hipError_t e;
    CamMats cm;
    // pv = projection * view, the matrix product phong.vert applies before model
    for (int c = 0; c < 4; ++c)
        for (int r = 0; r < 4; ++r) {
            float acc = cam.projection[0 * 4 + r] * cam.view[c * 4 + 0];
            acc = acc + cam.projection[1 * 4 + r] * cam.view[c * 4 + 1];
            acc = acc + cam.projection[2 * 4 + r] * cam.view[c * 4 + 2];
            acc = acc + cam.projection[3 * 4 + r] * cam.view[c * 4 + 3];
            cm.pv[c * 4 + r] = acc;
        }
    cm.W = cam.width;
    cm.H = cam.height;
    cm.cull = cam.cull_back;
    const size_t nslots = (size_t)sc.ntri * 2;
    hipLaunchKernelGGL(k_gbuf_setup, dim3(setup_blocks(sc.ntri, (size_t)cam.width * cam.height * 2)), dim3(256), 0, s,
                       sc, cm, rs.rec, rs.attr, rs.counts, rs.bcounts, (uint32_t *)vis);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (sc.ntri > 0) {
        if ((e = raster_scan(rs, nslots, true, s)) != hipSuccess) return e;
        GbufFrag f{rs.attr, (unsigned long long *)vis, cam.width};
        hipLaunchKernelGGL(k_raster_items<GbufFrag>, dim3(raster_grid<GbufFrag, false>()), dim3(256), 0, s, rs.rec, rs.offs,
                           rs.chunk, rs.chunk_cap, (int)nslots, f);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        GbufBlockFrag fb{rs.attr, (unsigned long long *)vis, cam.width, cam.height};
        hipLaunchKernelGGL(k_raster_blocks<GbufBlockFrag>, dim3(kRasterBlocks), dim3(256), 0, s, rs.rec, rs.boffs,
                           rs.bchunk, rs.chunk_cap, (int)nslots, fb);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    dim3 grid((cam.width + 15) / 16, (cam.height + 15) / 16);
    hipLaunchKernelGGL(k_gbuf_resolve, grid, dim3(256), 0, s, sc, cm, (const unsigned long long *)vis, gbuf);
    return hipGetLastError();
}

}  // namespace vctk
