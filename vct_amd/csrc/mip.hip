// mip.hip -- the radiance mip chain (filterRadiance.comp KERNEL_BOX2,
// src/Application.cpp:877-921) fused over three levels per launch.
//
// The reference dispatches one compute pass per level with a full barrier in
// between, re-reading each level from memory.  Here a launch takes 8^3 regions
// of the source level (two 4^3 bricks per axis, contiguous 1 KB brick runs) and
// produces the 4^3, 2^3 and 1^3 blocks of the next three levels: a wavefront per
// region where the source has one face (k_mip_regions), a workgroup where it has
// six or is smaller than a region (k_mip_chain).  So level 0 -- the only large one
// -- is read exactly once.  Each level is rounded to its storage format before the
// next one is filtered from it, exactly as a per-level pass over stored texels would
// be, and the eight taps are summed in the reference's offset order, so the chain is
// bit-identical to filtering level by level.
//
// Anisotropic chains keep six directional volumes per level >= 1 (+x,-x,+y,
// -y,+z,-z): each is the mean of the four front-to-back composites
// near + (1 - near.a) * far of the child pairs along that axis.
#pragma clang fp contract(off)

#include "vct_device.h"

namespace vctk {

struct MipArgs {
    char *pyr;
    LevelInfo src;
    LevelInfo out[3];
    int nout;
    int fp32;  // stage format: 1 = fp32x4, 0 = fp16 pairs
    // source level 0 only: its bricks known to hold +0 (PyrDesc::zero0), or null
    const uint8_t *zero0;
};

// Whether brick (x, y, z) >> 2 of the source is known to hold +0: its texels
// are then not read.
__device__ __forceinline__ bool src_zero(const MipArgs &a, int x, int y, int z) {
    if (a.zero0 == nullptr) return false;
    const uint32_t nb = (uint32_t)a.src.nb;
    return (a.zero0[((uint32_t)(z >> 2) * nb + (uint32_t)(y >> 2)) * nb + (uint32_t)(x >> 2)] & 1u) != 0;
}

__device__ __forceinline__ float4 round_stage(float4 v, int fp32) {
    if (fp32) return v;
    return make_float4(q16(v.x), q16(v.y), q16(v.z), q16(v.w));
}

// One filtering step of the chain: the (cur/2)^3 texels per face of output
// level k from the cur^3 texels per face in LDS (as many source faces as outputs).
// CUR: cur as a compile-time constant (0: use the argument), which turns the
// index arithmetic into shifts.
template <bool ANISO, int CUR>
__device__ __forceinline__ void mip_step(const MipArgs &a, int cur_rt, const float4 *in, int in_stride,
                                         float4 *out, int out_stride, int k, int ox, int oy, int oz) {
    constexpr int NF = ANISO ? 6 : 1;
    const int cur = CUR ? CUR : cur_rt;
    const int d = cur >> 1;
    const LevelInfo &ol = a.out[k];
    const int sh = k + 1;
    const int gx = ox >> sh, gy = oy >> sh, gz = oz >> sh;
    const int d3 = d * d * d;
    for (int i = threadIdx.x; i < d3 * NF; i += 256) {
        const int f = i / d3;
        const int vi = i - f * d3;
        const int x = vi % d, y = (vi / d) % d, z = vi / (d * d);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!ANISO) {
            // BOX2 offsets in filterRadiance.comp order: (0,0,0),(0,0,1),(0,1,0),(0,1,1),(1,0,0),...
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int dx = (o >> 2) & 1, dy = (o >> 1) & 1, dz = o & 1;
                const float4 t = in[((2 * z + dz) * cur + (2 * y + dy)) * cur + (2 * x + dx)];
                v.x = v.x + t.x;
                v.y = v.y + t.y;
                v.z = v.z + t.z;
                v.w = v.w + t.w;
            }
            v.x = v.x * 0.125f;
            v.y = v.y * 0.125f;
            v.z = v.z * 0.125f;
            v.w = v.w * 0.125f;
        } else {
            const int ax = f >> 1, neg = f & 1;
            const float4 *src = in + (size_t)f * in_stride;
            const int oa = ax == 0 ? 1 : 0, ob = ax == 2 ? 1 : 2;
#pragma unroll
            for (int pa = 0; pa < 2; ++pa)
#pragma unroll
                for (int pb = 0; pb < 2; ++pb) {
                    int cn[3] = {2 * x, 2 * y, 2 * z}, cf[3] = {2 * x, 2 * y, 2 * z};
                    cn[oa] += pa;
                    cf[oa] += pa;
                    cn[ob] += pb;
                    cf[ob] += pb;
                    cn[ax] += neg ? 1 : 0;
                    cf[ax] += neg ? 0 : 1;
                    const float4 pn = src[(cn[2] * cur + cn[1]) * cur + cn[0]];
                    const float4 pf = src[(cf[2] * cur + cf[1]) * cur + cf[0]];
                    const float t = 1.0f - pn.w;
                    v.x = v.x + (pn.x + t * pf.x);
                    v.y = v.y + (pn.y + t * pf.y);
                    v.z = v.z + (pn.z + t * pf.z);
                    v.w = v.w + (pn.w + t * pf.w);
                }
            v.x = v.x * 0.25f;
            v.y = v.y * 0.25f;
            v.z = v.z * 0.25f;
            v.w = v.w * 0.25f;
        }
        v = round_stage(v, a.fp32);
        out[(size_t)f * out_stride + vi] = v;
        store_stage_texel(a.pyr, ol, gx + x, gy + y, gz + z, NF == 6 ? f : 0, v);
    }
}

// The first step of an 8^3 region (4^3 texels per face): wavefront w filters
// faces w and w + 4, one texel per lane.  The face is wave-uniform, so the
// child offsets of its near/far pairs are scalar values and only the texel's
// base address is per lane.  Same taps, in the same order, as mip_step.
__device__ __forceinline__ void mip_step8(const MipArgs &a, const float4 *in, float4 *out, int ox, int oy, int oz) {
    constexpr int NF = 6;
    constexpr int cur = 8;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int x = lane & 3, y = (lane >> 2) & 3, z = lane >> 4;
    const int base = ((2 * z) * cur + 2 * y) * cur + 2 * x;
    const LevelInfo &ol = a.out[0];
    for (int f = w; f < NF; f += 4) {
        const float4 *c = in + f * 512 + base;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        const int ax = f >> 1, neg = f & 1;
        // strides of the face's axis and of the two axes across it (oa, ob
        // as in mip_step: y, z for x; x, z for y; x, y for z)
        const int s_ax = ax == 0 ? 1 : (ax == 1 ? cur : cur * cur);
        const int s_oa = ax == 0 ? cur : 1;
        const int s_ob = ax == 2 ? cur : cur * cur;
        const int near = neg ? s_ax : 0, far = neg ? 0 : s_ax;
#pragma unroll
        for (int pa = 0; pa < 2; ++pa)
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) {
                const int o = pa * s_oa + pb * s_ob;
                const float4 pn = c[o + near];
                const float4 pf = c[o + far];
                const float t = 1.0f - pn.w;
                v.x = v.x + (pn.x + t * pf.x);
                v.y = v.y + (pn.y + t * pf.y);
                v.z = v.z + (pn.z + t * pf.z);
                v.w = v.w + (pn.w + t * pf.w);
            }
        v.x = v.x * 0.25f;
        v.y = v.y * 0.25f;
        v.z = v.z * 0.25f;
        v.w = v.w * 0.25f;
        v = round_stage(v, a.fp32);
        out[f * 64 + lane] = v;
        store_stage_texel(a.pyr, ol, (ox >> 1) + x, (oy >> 1) + y, (oz >> 1) + z, f, v);
    }
}

// ANISO: source and outputs have six faces.  Without, the source is a level of 2^3
// or 4^3 texels (a larger one goes to k_mip_regions).  LDS: the 8^3 source region
// (per face), then the ping-pong buffers of the three output steps (4^3, 2^3, 1^3
// per face).
template <bool ANISO>
__global__ __launch_bounds__(256) void k_mip_chain(MipArgs a) {
    constexpr int NF = ANISO ? 6 : 1;
    __shared__ float4 bufA[NF][ANISO ? 512 : 64];
    __shared__ float4 bufB[NF][64];
    const int tid = threadIdx.x;
    const int s = a.src.size;
    const int R = s < 8 ? s : 8;
    const int nreg = s / R;
    // XCD-aware order: workgroup b runs on XCD b % 8, so give each XCD a
    // contiguous run of regions; x-neighbours then share an L2 and run at
    // about the same time, which merges the two halves of the pair elements
    // on a region's x boundary in one L2 line before it is written back.
    const int nblk = nreg * nreg * nreg;
    const int b = (nblk & 7) == 0 ? (int)(blockIdx.x & 7u) * (nblk >> 3) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const int rx = b % nreg, ry = (b / nreg) % nreg, rz = b / (nreg * nreg);
    const int ox = rx * R, oy = ry * R, oz = rz * R;
    const int R3 = R * R * R;
    for (int f = 0; f < NF; ++f) {
        if (ANISO && R == 8 && !a.fp32) {
            // fp16 pairs: the elements of even x hold texels x and x+1; walk
            // brick by brick (32 such elements per brick)
            const int i = tid;  // 256 threads, 256 pair elements
            const int j = i >> 5, v = i & 31;
            const int x = ox + (j & 1) * 4 + (v & 1) * 2;
            const int y = oy + ((j >> 1) & 1) * 4 + ((v >> 1) & 3);
            const int z = oz + (j >> 2) * 4 + (v >> 3);
            const uint4 e = *(const uint4 *)(a.pyr + a.src.stage + (size_t)elem_index(a.src, x, y, z, f) * 16);
            float4 *d = &bufA[f][((z - oz) * R + (y - oy)) * R + (x - ox)];
            d[0] = unpack_h4(e.x, e.y);
            d[1] = unpack_h4(e.z, e.w);
        } else {
            for (int i = tid; i < R3; i += 256) {
                int x, y, z;
                if (ANISO && R == 8) {  // brick-major walk: 8 bricks of 64 contiguous voxels
                    const int j = i >> 6, v = i & 63;
                    x = ox + (j & 1) * 4 + (v & 3);
                    y = oy + ((j >> 1) & 1) * 4 + ((v >> 2) & 3);
                    z = oz + (j >> 2) * 4 + (v >> 4);
                } else {
                    x = i % R;
                    y = (i / R) % R;
                    z = i / (R * R);
                }
                bufA[f][((z - oz) * R + (y - oy)) * R + (x - ox)] = load_stage_texel(a.pyr, a.src, x, y, z, f);
            }
        }
    }
    __syncthreads();
    if (ANISO && R == 8) {  // the three steps with their sizes known at compile time
        mip_step8(a, &bufA[0][0], &bufB[0][0], ox, oy, oz);
        if (a.nout > 1) {
            __syncthreads();
            mip_step<ANISO, 4>(a, 4, &bufB[0][0], 64, &bufA[0][0], 8, 1, ox, oy, oz);
        }
        if (a.nout > 2) {
            __syncthreads();
            mip_step<ANISO, 2>(a, 2, &bufA[0][0], 8, &bufB[0][0], 64, 2, ox, oy, oz);
        }
        return;
    }
    int cur = R;
    float4 *in = &bufA[0][0];
    int in_stride = ANISO ? 512 : 64;
    for (int k = 0; k < a.nout; ++k) {
        const int d = cur >> 1;
        if (d < 1) break;
        // ping-pong: outputs of step k go to bufB (k even, <= 4^3 per face) or
        // bufA (k odd, <= 2^3 per face)
        float4 *out = (k & 1) ? &bufA[0][0] : &bufB[0][0];
        const int out_stride = (k & 1) ? 8 : 64;
        mip_step<ANISO, 0>(a, cur, in, in_stride, out, out_stride, k, ox, oy, oz);
        __syncthreads();
        in = out;
        in_stride = out_stride;
        cur = d;
    }
}

// One wavefront per 8^3 region of a source with one face, one output texel per
// lane: the lane loads its eight children (four pair elements, or eight fp32
// texels) and filters all its faces in registers; the two smaller steps go
// through LDS within the wavefront.  Same taps, in the same order, as mip_step.
//
// What bounds it: memory (1 KB read per brick that is not zero, 16 bytes written
// per texel and face).  With a workgroup per region, the children in LDS and a
// barrier before each step, three of four wavefronts waited in the isotropic
// steps and a CU had 8 regions in flight: the chain of 512^3 461 us, now 308;
// 256^3 with six faces 113, 110 (both at 3.3 TB/s beside the albedo chain); 128^3
// 13.8, 9.4.  Not storing zeros over zeros again (a record per region) gained
// nothing: two thirds of the regions of a 256^3 scene hold something.
template <bool ANISO, int CUR>
__device__ __forceinline__ float4 mip_wave_texel(const float4 *in, int f, int x, int y, int z) {
    const float4 *c = in + ((2 * z) * CUR + 2 * y) * CUR + 2 * x;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!ANISO) {
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            const float4 t = c[((o & 1) * CUR + ((o >> 1) & 1)) * CUR + (o >> 2)];
            v.x = v.x + t.x;
            v.y = v.y + t.y;
            v.z = v.z + t.z;
            v.w = v.w + t.w;
        }
        return make_float4(v.x * 0.125f, v.y * 0.125f, v.z * 0.125f, v.w * 0.125f);
    }
    const int ax = f >> 1, neg = f & 1;
    const int s_ax = ax == 0 ? 1 : (ax == 1 ? CUR : CUR * CUR);  // strides as in mip_step8
    const int s_oa = ax == 0 ? CUR : 1;
    const int s_ob = ax == 2 ? CUR : CUR * CUR;
    const int near = neg ? s_ax : 0, far = neg ? 0 : s_ax;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int o = (p >> 1) * s_oa + (p & 1) * s_ob;
        const float4 pn = c[o + near];
        const float4 pf = c[o + far];
        const float t = 1.0f - pn.w;
        v.x = v.x + (pn.x + t * pf.x);
        v.y = v.y + (pn.y + t * pf.y);
        v.z = v.z + (pn.z + t * pf.z);
        v.w = v.w + (pn.w + t * pf.w);
    }
    return make_float4(v.x * 0.25f, v.y * 0.25f, v.z * 0.25f, v.w * 0.25f);
}

template <bool ANISO, bool FP32>
__global__ __launch_bounds__(256) void k_mip_regions(MipArgs a) {
    constexpr int NF = ANISO ? 6 : 1;
    __shared__ float4 buf1[4][NF][64], buf2[4][NF][8];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nreg = (uint32_t)a.src.size >> 3;  // a power of two, as every level's size
    const int lg = __builtin_ctz(nreg);
    // XCD-aware order: workgroup b runs on XCD b % 8, so give each XCD a
    // contiguous run of regions; x-neighbours then share an L2 and run at
    // about the same time, which merges the two halves of the pair elements
    // on a region's x boundary in one L2 line before it is written back.
    const uint32_t nblk = gridDim.x;
    const uint32_t b = (nblk & 7u) == 0 ? (blockIdx.x & 7u) * (nblk >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const uint32_t r = b * 4u + (uint32_t)w;
    if (r >= nreg * nreg * nreg) return;  // no barrier below
    const int ox = (int)(r & (nreg - 1)) * 8, oy = (int)((r >> lg) & (nreg - 1)) * 8, oz = (int)(r >> (2 * lg)) * 8;
    const int X = lane & 3, Y = (lane >> 2) & 3, Z = lane >> 4;
    const int x = ox + 2 * X, y = oy + 2 * Y, z = oz + 2 * Z;  // the lane's children lie in one brick
    const bool zero = src_zero(a, x, y, z);
    const bool none = __ballot(!zero) == 0;
    float4 c[8];  // child (dx, dy, dz) = bits (2, 1, 0)
#pragma unroll
    for (int o = 0; o < 8; ++o) c[o] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!zero) {
        const char *p = a.pyr + a.src.stage + (size_t)elem_index(a.src, x, y, z, 0) * 16;
        if (FP32) {
#pragma unroll
            for (int o = 0; o < 8; ++o)
                c[o] = *(const float4 *)(p + ((o >> 2) + ((o >> 1) & 1) * 4 + (o & 1) * 16) * 16);
        } else {  // the element of an even x holds texels x and x + 1
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                const uint4 e = *(const uint4 *)(p + (((o >> 1) & 1) * 4 + (o & 1) * 16) * 16);
                c[o] = unpack_h4(e.x, e.y);
                c[4 + o] = unpack_h4(e.z, e.w);
            }
        }
    }
    const LevelInfo &ol = a.out[0];
    const int gx = (ox >> 1) + X, gy = (oy >> 1) + Y, gz = (oz >> 1) + Z;  // a region's outputs are one brick
    char *const q = a.pyr + ol.stage + (size_t)elem_index(ol, gx, gy, gz, 0) * 16;
    const uint32_t ql = ol.stage + elem_index(ol, gx - 1, gy, gz, 0) * 16u;  // wraps below 0 at gx = 0
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (none) {
            // zeros filter to +0
        } else if (!ANISO) {
            // BOX2 offsets in filterRadiance.comp order: (0,0,0),(0,0,1),(0,1,0),(0,1,1),(1,0,0),...
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                v.x = v.x + c[o].x;
                v.y = v.y + c[o].y;
                v.z = v.z + c[o].z;
                v.w = v.w + c[o].w;
            }
            v = make_float4(v.x * 0.125f, v.y * 0.125f, v.z * 0.125f, v.w * 0.125f);
        } else {
            const int ax = f >> 1, neg = f & 1;
            const int b_ax = 4 >> ax;                             // the bits of c's index: the face's axis
            const int b_oa = ax == 0 ? 2 : 4, b_ob = ax == 2 ? 2 : 1;  // and the two across it
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int o = (k >> 1 ? b_oa : 0) | (k & 1 ? b_ob : 0);
                const float4 pn = c[o | (neg ? b_ax : 0)], pf = c[o | (neg ? 0 : b_ax)];
                const float t = 1.0f - pn.w;
                v.x = v.x + (pn.x + t * pf.x);
                v.y = v.y + (pn.y + t * pf.y);
                v.z = v.z + (pn.z + t * pf.z);
                v.w = v.w + (pn.w + t * pf.w);
            }
            v = make_float4(v.x * 0.25f, v.y * 0.25f, v.z * 0.25f, v.w * 0.25f);
        }
        v = round_stage(v, FP32);
        if (!none) buf1[w][f][lane] = v;
        if (FP32) {
            *(float4 *)(q + f * 1024) = v;
        } else {
            // the lane's element: its texel and the next one in x, which the next
            // region stores for the last
            const uint2 h = pack_h4(v);
            const uint2 n = make_uint2(__shfl_down(h.x, 1, 64), __shfl_down(h.y, 1, 64));
            if (X < 3) *(uint4 *)(q + f * 1024) = make_uint4(h.x, h.y, n.x, n.y);
            else *(uint2 *)(q + f * 1024) = h;
            if (X == 0) *(uint2 *)(a.pyr + (uint32_t)(ql + f * 1024u) + 8) = h;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (a.nout > 1 && lane < 8 * NF) {
        const int f = lane >> 3, vi = lane & 7;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!none) v = round_stage(mip_wave_texel<ANISO, 4>(buf1[w][f], f, vi & 1, (vi >> 1) & 1, vi >> 2), FP32);
        buf2[w][f][vi] = v;
        store_stage_texel(a.pyr, a.out[1], (ox >> 2) + (vi & 1), (oy >> 2) + ((vi >> 1) & 1), (oz >> 2) + (vi >> 2), f, v);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (a.nout > 2 && lane < NF) {
        const float4 v = round_stage(mip_wave_texel<ANISO, 2>(buf2[w][lane], lane, 0, 0, 0), FP32);
        store_stage_texel(a.pyr, a.out[2], ox >> 3, oy >> 3, oz >> 3, lane, v);
    }
}

// FP8 E4M3 encode of one level: one 64-thread wavefront per (brick, face);
// the scale is the largest magnitude in the brick over 448 (1 if all zero).
// The chain is done with the level's stage by now, so the decoded texels
// (code * scale, what load_texel returns) take its place as fp32 elements,
// with zeros in the border element of texel -1 (the second half of which held
// texel 0 of an fp16 pair): the trace reads a texel with one 16-byte load and
// no decoding, which it would otherwise repeat for every corner of every
// sample.
__global__ __launch_bounds__(64) void k_fp8_encode(char *pyr, float *scales, LevelInfo L) {
    const int bf = blockIdx.x;  // brick * nfaces + face
    const int b = bf / L.nfaces, f = bf % L.nfaces;
    const int v = threadIdx.x;
    const int nb = L.nb;
    const int bx = b % nb, by = (b / nb) % nb, bz = b / (nb * nb);
    const int x = bx * 4 + (v & 3), y = by * 4 + ((v >> 2) & 3), z = bz * 4 + (v >> 4);
    const bool valid = x < L.size && y < L.size && z < L.size;
    float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) c = load_stage_texel(pyr, L, x, y, z, f);
    float m = fmaxf(fmaxf(__builtin_fabsf(c.x), __builtin_fabsf(c.y)), fmaxf(__builtin_fabsf(c.z), __builtin_fabsf(c.w)));
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    const float sc = m > 0.0f ? m / 448.0f : 1.0f;
    const uint32_t e = elem_index(L, x, y, z, f);  // brick and face: e / 64 (every stride is a multiple of 64)
    if (v == 0) scales[L.scale + (e >> 6)] = sc;
    const uint32_t code = f2fp8(c.x / sc) | (f2fp8(c.y / sc) << 8) | (f2fp8(c.z / sc) << 16) | (f2fp8(c.w / sc) << 24);
    *(uint32_t *)(pyr + L.base + (size_t)e * 4) = code;
    *(float4 *)(pyr + L.stage + (size_t)e * 16) = decode_fp8x4(code, sc);
    if (x == 0)  // the element index of x = -1 wraps below 0: the byte offset is formed in 32 bits
        *(float4 *)(pyr + (uint32_t)(L.stage + elem_index(L, -1, y, z, f) * 16u)) = make_float4(0.f, 0.f, 0.f, 0.f);
}

// ---------------------------------------------------------------- albedo chain
// The voxelColor chain of the same mipmap pass (Application.cpp:904-917): BOX2
// on an RGBA8 image, so every level is stored as packUnorm4x8 of the mean of
// its eight children read back as k/255 (filterRadiance.comp:14-65 with
// rgba8 image bindings).  Levels >= 1 are linear, x fastest.  Levels 1 and 2
// come from k_albedo_bricks (below); the coarser ones from k_albedo_chain,
// the region scheme of k_mip_chain: a workgroup loads an 8^3 region of a
// linear source level and writes up to three levels from LDS.
struct AlbedoMipArgs {
    const uint32_t *src;
    int src_size;
    uint32_t *out[3];
    int nout;
};

__global__ __launch_bounds__(256) void k_albedo_chain(AlbedoMipArgs a) {
    __shared__ float4 bufA[512];
    __shared__ float4 bufB[64];
    const int tid = threadIdx.x;
    const int s = a.src_size;
    const int R = s < 8 ? s : 8;
    const int nreg = s / R;
    const int b = (int)blockIdx.x;
    const int ox = (b % nreg) * R, oy = ((b / nreg) % nreg) * R, oz = (b / (nreg * nreg)) * R;
    const int R3 = R * R * R;
    for (int i = tid; i < R3; i += 256) {
        const int x = ox + i % R, y = oy + (i / R) % R, z = oz + i / (R * R);
        const uint32_t w = a.src[((size_t)z * s + y) * s + x];
        bufA[((z - oz) * R + (y - oy)) * R + (x - ox)] = make_float4(unorm8(w, 0), unorm8(w, 1), unorm8(w, 2),
                                                                     unorm8(w, 3));
    }
    __syncthreads();
    int cur = R;
    float4 *in = bufA;
    for (int k = 0; k < a.nout; ++k) {
        const int d = cur >> 1;
        if (d < 1) break;
        float4 *out = (k & 1) ? bufA : bufB;
        const int os = s >> (k + 1);  // output level size
        const int gx = ox >> (k + 1), gy = oy >> (k + 1), gz = oz >> (k + 1);
        for (int i = tid; i < d * d * d; i += 256) {
            const int x = i % d, y = (i / d) % d, z = i / (d * d);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            // BOX2 offsets in filterRadiance.comp order: (0,0,0),(0,0,1),(0,1,0),(0,1,1),(1,0,0),...
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int dx = (o >> 2) & 1, dy = (o >> 1) & 1, dz = o & 1;
                const float4 t = in[((2 * z + dz) * cur + (2 * y + dy)) * cur + (2 * x + dx)];
                v.x = v.x + t.x;
                v.y = v.y + t.y;
                v.z = v.z + t.z;
                v.w = v.w + t.w;
            }
            const uint32_t pw = pack_unorm4x8(v.x * 0.125f, v.y * 0.125f, v.z * 0.125f, v.w * 0.125f);
            a.out[k][((size_t)(gz + z) * os + (gy + y)) * os + (gx + x)] = pw;
            out[i] = make_float4(unorm8(pw, 0), unorm8(pw, 1), unorm8(pw, 2), unorm8(pw, 3));
        }
        __syncthreads();
        in = out;
        cur = d;
    }
}

// Levels 1 and 2 of the albedo chain straight from the bricked grid: one
// thread per 4^3 brick, which holds exactly the 2^3 level-1 texels and the one
// level-2 texel it filters to.  The brick is read a z-slab pair at a time
// (eight 16-byte loads of 32 words), every level-1 texel is rounded to RGBA8
// before level 2 is filtered from it, and the taps are summed in the BOX2
// order of filterRadiance.comp -- the same values as filtering level by level.
__global__ __launch_bounds__(256) void k_albedo_bricks(const uint32_t *__restrict__ grid,
                                                       const uint8_t *__restrict__ zero0, int dim, uint32_t *out1,
                                                       uint32_t *out2) {
    const int nb = dim >> 2;
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= (uint32_t)nb * nb * nb) return;
    const int lg = __builtin_ctz((unsigned)nb);
    const int bx = (int)(b & (uint32_t)(nb - 1)), by = (int)((b >> lg) & (uint32_t)(nb - 1)), bz = (int)(b >> (2 * lg));
    if (zero0 != nullptr && (zero0[b] & 2u) != 0) {  // bit 1: every word of the brick is 0
        // every word of the brick is 0: the texels it filters to are
        // packUnorm4x8 of sums of zeros, 0, and the brick is not read
        const int s1 = dim >> 1;
#pragma unroll
        for (int cz = 0; cz < 2; ++cz)
#pragma unroll
            for (int cy = 0; cy < 2; ++cy)
                *(uint2 *)&out1[((size_t)(bz * 2 + cz) * s1 + (by * 2 + cy)) * s1 + bx * 2] = make_uint2(0u, 0u);
        if (out2 != nullptr) {
            const int s2 = dim >> 2;
            out2[((size_t)bz * s2 + by) * s2 + bx] = 0u;
        }
        return;
    }
    const uint4 *src = (const uint4 *)(grid + ((size_t)b << 6));
    const int s1 = dim >> 1;
    float4 l1[8];  // the rounded level-1 texels, (cx, cy, cz) = bits (2, 1, 0) in BOX2 order
#pragma unroll
    for (int cz = 0; cz < 2; ++cz) {
        uint32_t w[32];  // z rows 2cz, 2cz+1 of the brick: w[(z & 1) * 16 + y * 4 + x]
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint4 v = src[cz * 8 + k];
            w[k * 4 + 0] = v.x;
            w[k * 4 + 1] = v.y;
            w[k * 4 + 2] = v.z;
            w[k * 4 + 3] = v.w;
        }
#pragma unroll
        for (int cy = 0; cy < 2; ++cy)
#pragma unroll
            for (int cx = 0; cx < 2; ++cx) {
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int o = 0; o < 8; ++o) {  // (0,0,0),(0,0,1),(0,1,0),(0,1,1),(1,0,0),...
                    const int dx = (o >> 2) & 1, dy = (o >> 1) & 1, dz = o & 1;
                    const uint32_t t = w[dz * 16 + (2 * cy + dy) * 4 + (2 * cx + dx)];
                    v.x = v.x + unorm8(t, 0);
                    v.y = v.y + unorm8(t, 1);
                    v.z = v.z + unorm8(t, 2);
                    v.w = v.w + unorm8(t, 3);
                }
                const uint32_t pw = pack_unorm4x8(v.x * 0.125f, v.y * 0.125f, v.z * 0.125f, v.w * 0.125f);
                const int x = bx * 2 + cx, y = by * 2 + cy, z = bz * 2 + cz;
                out1[((size_t)z * s1 + y) * s1 + x] = pw;
                l1[(cx << 2) | (cy << 1) | cz] = make_float4(unorm8(pw, 0), unorm8(pw, 1), unorm8(pw, 2), unorm8(pw, 3));
            }
    }
    if (out2 == nullptr) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        v.x = v.x + l1[o].x;
        v.y = v.y + l1[o].y;
        v.z = v.z + l1[o].z;
        v.w = v.w + l1[o].w;
    }
    const int s2 = dim >> 2;
    out2[((size_t)bz * s2 + by) * s2 + bx] = pack_unorm4x8(v.x * 0.125f, v.y * 0.125f, v.z * 0.125f, v.w * 0.125f);
}

hipError_t launch_albedo_chain(const uint32_t *grid, const uint8_t *zero0, uint32_t *const *levels, int dim, int nlevels,
                               hipStream_t s) {
    if (nlevels < 2) return hipSuccess;
    {
        const unsigned nbricks = (unsigned)((dim >> 2) * (dim >> 2) * (dim >> 2));
        hipLaunchKernelGGL(k_albedo_bricks, dim3((nbricks + 255) / 256), dim3(256), 0, s, grid, zero0, dim, levels[1],
                           nlevels > 2 ? levels[2] : nullptr);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    int src = nlevels > 2 ? 2 : 1;
    while (src + 1 < nlevels) {
        const int size = dim >> src;
        const int R = size < 8 ? size : 8;
        if (R < 2) break;
        const int lg = R == 8 ? 3 : (R == 4 ? 2 : 1);
        int nout = nlevels - 1 - src;
        if (nout > lg) nout = lg;
        AlbedoMipArgs a;
        a.src = levels[src];
        a.src_size = size;
        for (int k = 0; k < 3; ++k) a.out[k] = levels[k < nout ? src + 1 + k : src + 1];
        a.nout = nout;
        const int nreg = size / R;
        hipLaunchKernelGGL(k_albedo_chain, dim3((unsigned)(nreg * nreg * nreg)), dim3(256), 0, s, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        src += nout;
    }
    return hipSuccess;
}

hipError_t launch_mip(const PyrDesc &pyr, hipStream_t s) {
    const int fp32 = pyr.storage == VCT_STORE_FP32 ? 1 : 0;
    int src = 0;
    while (src + 1 < pyr.nlevels) {
        const LevelInfo &S = pyr.lv[src];
        const int R = S.size < 8 ? S.size : 8;
        if (R < 2) break;
        const int lg = R == 8 ? 3 : (R == 4 ? 2 : 1);
        int nout = pyr.nlevels - 1 - src;
        if (nout > lg) nout = lg;
        MipArgs a;
        a.pyr = pyr.pyr;
        a.src = S;
        for (int k = 0; k < 3; ++k) a.out[k] = pyr.lv[k < nout ? src + 1 + k : src + 1];
        a.nout = nout;
        a.fp32 = fp32;
        a.zero0 = src == 0 ? pyr.zero0 : nullptr;
        const int nreg = S.size / R;
        dim3 grid((unsigned)(nreg * nreg * nreg));
        const dim3 wgrid((grid.x + 3) / 4);  // a wavefront per region
        if (R == 8 && S.nfaces == 1 && pyr.aniso) {
            if (fp32) hipLaunchKernelGGL((k_mip_regions<true, true>), wgrid, dim3(256), 0, s, a);
            else hipLaunchKernelGGL((k_mip_regions<true, false>), wgrid, dim3(256), 0, s, a);
        } else if (R == 8 && S.nfaces == 1) {
            if (fp32) hipLaunchKernelGGL((k_mip_regions<false, true>), wgrid, dim3(256), 0, s, a);
            else hipLaunchKernelGGL((k_mip_regions<false, false>), wgrid, dim3(256), 0, s, a);
        } else if (pyr.aniso) hipLaunchKernelGGL(k_mip_chain<true>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_mip_chain<false>, grid, dim3(256), 0, s, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        src += nout;
    }
    if (pyr.storage == VCT_STORE_FP8) {
        for (int l = 3; l < pyr.nlevels; ++l) {
            const LevelInfo &L = pyr.lv[l];
            hipLaunchKernelGGL(k_fp8_encode, dim3((unsigned)(L.nb * L.nb * L.nb * L.nfaces)), dim3(64), 0, s, pyr.pyr,
                               pyr.scales, L);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

}  // namespace vctk
