// trace.hip -- the cone-traced indirect light of phong.frag: traceCone
// (shaders/phong.frag:135-180), the 6-cone diffuse gather with its occlusion
// term and the specular cone (:455-512).
//
// The sampler and the per-pixel gather live in trace_core.h.
#include "trace_core.h"

namespace vctk {

// Runs of consecutive workgroups on one XCD: workgroup b runs on XCD b % 8, and
// neighbouring tiles share bricks in its L2, while every XCD gets parts of the
// whole image (one contiguous eighth each left some XCDs idle at the end: the
// 1001x567 FP32 gather took 266 us instead of 163).
constexpr int kTraceRun = 4, kSplitRun = 16;
__device__ __forceinline__ int xcd_group(int run) {
    const int j = (int)(blockIdx.x >> 3);
    return ((j / run) * 8 + (int)(blockIdx.x & 7u)) * run + j % run;
}

// A workgroup is a 16x16 pixel tile of four 8x8 wavefront tiles: its
// wavefronts march neighbouring cones through the same bricks at about the same
// time, which the scalar data cache they share rewards (a workgroup whose
// wavefronts take different cones of one tile misses it three times as often).
// Six wavefronts per SIMD (five for the formats of one texel per element) at
// the price of registers kept in scratch between cones (with six directions 16 to
// 27 of a lane's, 64 to 96 bytes; isotropic at most 6): 490 -> 467 us for the
// 1280x720 six-direction gather, though 158 of the 225 MB that a 1920x1080 launch
// writes are scratch.  With reflections the grid holds every tile
// twice, first its specular cones (the longer and less even half), then its
// diffuse cones: shorter wavefronts leave a shorter tail (574 -> 529 us for that
// gather by itself).  The whole of it, against one contiguous band of tiles per
// XCD, five wavefronts per SIMD and addresses formed before the zero test:
// 509 -> 453 us there, 1.35 -> 1.20 ms at 1920x1080.
template <int MODE, bool ANISO, bool WARP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == 0 ? 6 : 5))) void k_trace(
    TraceLaunch t, PyrArgs pa, int tiles_x, int tiles) {
    int tile = xcd_group(kTraceRun);
    const bool spec = t.enable_reflections && tile < tiles;
    if (!spec && t.enable_reflections) tile -= tiles;
    if (tile >= tiles) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int px = (tile % tiles_x) * 16 + (wave & 1) * 8 + (lane & 7);
    const int py = (tile / tiles_x) * 16 + (wave >> 1) * 8 + (lane >> 3);
    if (px >= t.width || py >= t.height) return;
    const size_t pi = (size_t)py * t.width + px;
    const __amdgpu_buffer_rsrc_t rs = pyr_rsrc(pa);
    TracePixel x;
    load_pixel(t, pi, x);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (spec) {
        if (x.covered) v = specular_cone<MODE, ANISO, WARP>(t, pa, rs, x);
        t.out_spec[pi] = v;
        return;
    }
    if (x.covered) {
        float4 sum = v;
        for (int c = 0; c < 6; ++c) add_cone(sum, diffuse_cone<MODE, ANISO, WARP>(t, pa, rs, x, c), c);
        v = indirect_value(t, sum);
    }
    t.out_ind[pi] = v;
}

// Small images: a workgroup is one 8x8 tile, its first `parts` wavefronts share
// the six diffuse cones (cone c by wavefront c % parts) and one more takes the
// specular cone.  The last diffuse wavefront to finish (LDS counter) adds the
// six results in order, so none waits for another and the sums are k_trace's.
// Where an image has fewer tiles than the chip holds wavefronts, a tile's time
// is the frame's: 64x64 to 256x256 took the same 62 us (room, isotropic), 147 us
// (objects, six directions) with one wavefront per tile, 25 us (17
// with six parts) and 79 us here.
template <int MODE, bool ANISO, bool WARP>
__global__ __launch_bounds__(448) __attribute__((amdgpu_waves_per_eu(MODE == 0 ? 6 : 5))) void k_trace_split(
    TraceLaunch t, PyrArgs pa, int tiles_x, int tiles, int parts) {
    __shared__ float4 part[6][64];
    __shared__ uint32_t done;
    const int tile = xcd_group(kSplitRun);
    if (tile >= tiles) return;
    if (threadIdx.x == 0) done = 0u;
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int px = (tile % tiles_x) * 8 + (lane & 7), py = (tile / tiles_x) * 8 + (lane >> 3);
    if (px >= t.width || py >= t.height) return;  // lane 0 is inside
    const size_t pi = (size_t)py * t.width + px;
    const __amdgpu_buffer_rsrc_t rs = pyr_rsrc(pa);
    TracePixel x;
    load_pixel(t, pi, x);
    if (wave == parts) {
        float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
        if (x.covered) r = specular_cone<MODE, ANISO, WARP>(t, pa, rs, x);
        t.out_spec[pi] = r;
        return;
    }
    if (x.covered) {
        for (int c = wave; c < 6; c += parts) part[c][lane] = diffuse_cone<MODE, ANISO, WARP>(t, pa, rs, x, c);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    uint32_t n = 0u;
    if (lane == 0) n = atomicAdd(&done, 1u);
    if (__builtin_amdgcn_readfirstlane(n) != (uint32_t)parts - 1u) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (x.covered) {
        float4 sum = v;
#pragma unroll
        for (int c = 0; c < 6; ++c) add_cone(sum, part[c][lane], c);
        v = indirect_value(t, sum);
    }
    t.out_ind[pi] = v;
}

hipError_t launch_trace(const PyrDesc &pyr, const TraceLaunch &t, hipStream_t s) {
    // k_trace_split where it is the faster one.  In us, launch after launch of one view,
    // k_trace / two / three parts (the room at 64^3, the 2,064 objects at 128^3), with a
    // specular cone: isotropic up to 8192 tiles, room 640x360 89 / 75 / 73, 960x540 153 /
    // 146 / 146, 1280x720 246 / 242 / 246, FP32 190 / 185 / 189 and 314 / 315 / 322 at the
    // last two, objects 640x360 141 / 122 / 126, 960x540 228 / 232 / 242; six directions up
    // to 4096, room 640x360 146 / 120 / 126, 720x405 168 / 146 / 152, objects 173 / 171 /
    // 180, 202 / 199 / 207, 960x540 296 / 306 / 319, FP32 640x360 213 / 215 / 222, 960x540
    // 372 / 389 / 409, FP8 186 / 190 / 196, 334 / 346 / 363.
    // Where launches of several views overlap, a longest tile costs less and the parts'
    // set-up more: k_trace is ahead by 1 to 4% at 1001x567 and above.  Without a specular
    // cone the warped six-direction kernel, which keeps most in scratch, still loses more
    // by its longest tile up to 9216 tiles (k_trace / two parts: 720x405 198 / 153, 960x540
    // 259 / 220, 1001x567 273 / 228; overlapping 94.6 / 93.3, 164.3 / 165.5), though no
    // longer at 1280x720 (overlapping 285.9 / 289.0).  Six parts, while six wavefronts per
    // tile leave SIMDs idle: room 128x128 isotropic 15 (three parts 22), 256x256 27 (26).
    const int tiles8 = ((t.width + 7) / 8) * ((t.height + 7) / 8);
    const bool split = tiles8 <= (!pyr.aniso ? 8192 : (t.warp && !t.enable_reflections ? 9216 : 4096));
    const int parts = pyr.aniso ? 2 : (!t.enable_reflections && tiles8 <= 512 ? 6 : 3);
    const int edge = split ? 8 : 16, run = split ? kSplitRun : kTraceRun;
    const int tiles_x = (t.width + edge - 1) / edge, tiles_y = (t.height + edge - 1) / edge;
    const int tiles = tiles_x * tiles_y;
    const int groups = split || !t.enable_reflections ? tiles : 2 * tiles;
    const dim3 grid((unsigned)((groups + 8 * run - 1) / (8 * run) * (8 * run)));
    const dim3 block(split ? 64 * (parts + (t.enable_reflections ? 1 : 0)) : 256);
    const int mode = pyr.storage == VCT_STORE_FP32 ? 1 : (pyr.storage == VCT_STORE_FP8 ? 2 : 0);
#define VCT_TRACE_LAUNCH(M, A, W)                                                                              \
    if (split)                                                                                                 \
        hipLaunchKernelGGL((k_trace_split<M, A, W>), grid, block, 0, s, t, pyr_args(pyr, t.nested), tiles_x, tiles, \
                           parts);                                                                             \
    else                                                                                                       \
        hipLaunchKernelGGL((k_trace<M, A, W>), grid, block, 0, s, t, pyr_args(pyr, t.nested), tiles_x, tiles)
#define VCT_TRACE_MODES(A, W)            \
    if (mode == 0) {                     \
        VCT_TRACE_LAUNCH(0, A, W);       \
    } else if (mode == 1) {              \
        VCT_TRACE_LAUNCH(1, A, W);       \
    } else {                             \
        VCT_TRACE_LAUNCH(2, A, W);       \
    }
    if (pyr.aniso && t.warp) {
        VCT_TRACE_MODES(true, true);
    } else if (pyr.aniso) {
        VCT_TRACE_MODES(true, false);
    } else if (t.warp) {
        VCT_TRACE_MODES(false, true);
    } else {
        VCT_TRACE_MODES(false, false);
    }
#undef VCT_TRACE_MODES
#undef VCT_TRACE_LAUNCH
    return hipGetLastError();
}

}  // namespace vctk
