// trace_core.h -- the cone tracer's device code: the pyramid sampler,
// traceCone (shaders/phong.frag:135-180) and the per-pixel gather of
// phong.frag:455-512.  Shared by the trace kernels (trace.hip) and the learned
// gather's per-tile fallback (learned.hip).
//
// Sampling restates the reference sampler (src/Application.h:144-146,
// Application.cpp:1094-1098): LINEAR_MIPMAP_LINEAR with the lambda clamp to
// the last level, trilinear inside a level, border (0,0,0,0) outside.
// Accumulation is FP32 whatever the storage format.
#pragma once

#include "vct_device.h"

namespace vctk {

// ---- trilinear sampling ------------------------------------------------------
// Every fetch is a buffer load through one descriptor that spans the whole
// pyramid (kept in scalar registers), with a 32-bit byte offset per lane.  An
// element index is a sum of per-axis terms (vct_internal.h):
//   X(x) = (x>>2)*sx + (x&3),  Y(y) = (y>>2)*sy + (y&3)*4,
//   Z(z) = (z>>2)*sz + (z&3)*16, plus 64 per face.
// Corners outside the level (the border) are read from the zero border bricks
// around every level, so all fetches are unconditional.  fp16 levels store
// texel pairs (x, x+1) per element: a trilinear sample is four 16-byte loads,
// one per (y, z) corner pair, instead of eight 8-byte loads -- the vector memory
// pipeline processes a wavefront's load in the same number of cycles for 8 or
// 16 bytes per lane, so this halves the trace's dominant cost.  fp32 levels, and
// fp8 levels in their decoded copy (LevelInfo::stage, written by the encoder),
// hold one 16-byte texel per element: eight loads.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// What the sampler needs of a level, by value in the kernel arguments: a level
// index is wave-uniform, so its fields are scalar loads whatever the kernel has
// stored before (behind a pointer the compiler has to load them per lane after
// the first store, and every product with them becomes vector work).
struct SampleLevel {
    float fs;             // edge length
    uint32_t org;         // byte offset of the level's storage (its first border brick)
    uint32_t sx, sy, sz;  // LevelInfo strides
    int nfaces;
    int one;              // one fp32 texel per element instead of an fp16 pair
    int pad;
};
struct PyrArgs {
    const char *pyr;
    uint32_t bytes;
    int dim, nlevels;
    int nested;  // TraceLaunch::nested
    SampleLevel lv[VCT_MAX_LEVELS];
};

__device__ __forceinline__ uint4 bload16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    return make_uint4(v.x, v.y, v.z, v.w);
}
// Scalar load of 16 bytes at a wave-uniform offset: through the constant
// address space the load becomes s_load_dwordx4 into SGPRs (scalar data cache,
// not the vector memory pipeline).  The pyramid is not written while a trace
// runs.  Nothing checks the offset (bload16's descriptor has the size): the callers'
// indices keep it inside the allocation.
typedef __attribute__((address_space(4))) const char cchar;
__device__ __forceinline__ uint4 sload16(const char *pyr, uint32_t off) {
    const u32x4 v = *(const __attribute__((address_space(4))) u32x4 *)((cchar *)pyr + off);
    return make_uint4(v.x, v.y, v.z, v.w);
}

// warp_sample (vct_device.h) for the march: at 1080p and above a wavefront's
// positions nearly always lie in one cell of the 32^3 texture, whose eight
// texels then come through scalar loads (the texture is not written while a
// trace runs); the per-lane form fetches eight float4 per step and lane.  The
// same products and sums in the same order, so both forms agree bit for bit.
__device__ __forceinline__ void warp_sample_march(const float4 *__restrict__ wm, float p[3]) {
    int i0[3], i1[3];
    float f[3];
    bool same = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float u = p[k] * (float)kWarpDim - 0.5f;
        const float fl = __builtin_floorf(u);
        f[k] = u - fl;
        const int a = (int)fl;
        same = same && __builtin_amdgcn_readfirstlane(a) == a;
        i0[k] = a < 0 ? 0 : (a > kWarpDim - 1 ? kWarpDim - 1 : a);
        i1[k] = a + 1 < 0 ? 0 : (a + 1 > kWarpDim - 1 ? kWarpDim - 1 : a + 1);
    }
    if (__ballot(same) != __ballot(true)) {
        warp_sample(wm, p, p);
        return;
    }
    float acc[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int dx = c & 1, dy = (c >> 1) & 1, dz = c >> 2;
        const float w = ((dx ? f[0] : 1.0f - f[0]) * (dy ? f[1] : 1.0f - f[1])) * (dz ? f[2] : 1.0f - f[2]);
        const uint32_t e = (uint32_t)(((dz ? i1[2] : i0[2]) * kWarpDim + (dy ? i1[1] : i0[1])) * kWarpDim +
                                      (dx ? i1[0] : i0[0]));
        const uint4 t = sload16((const char *)wm, __builtin_amdgcn_readfirstlane(e) * 16u);
        acc[0] = acc[0] + w * __uint_as_float(t.x);
        acc[1] = acc[1] + w * __uint_as_float(t.y);
        acc[2] = acc[2] + w * __uint_as_float(t.z);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = acc[k];
}

// All texels of a uniform fetch are +0 (empty space): their weighted sum adds
// exactly 0, so the weighting is skipped.  The test runs on the scalar unit,
// beside the vector work of the other wavefronts.
template <int N>
__device__ __forceinline__ bool zero16(const uint4 (&v)[N]) {
    uint32_t o = 0u;
#pragma unroll
    for (int c = 0; c < N; ++c) o |= (v[c].x | v[c].y) | (v[c].z | v[c].w);
    return o == 0u;
}

__device__ __forceinline__ uint64_t or16(const uint4 &v) {
    return ((uint64_t)v.y << 32 | v.x) | ((uint64_t)v.w << 32 | v.z);
}

__device__ __forceinline__ float hlo(uint32_t v) { return __half2float(__ushort_as_half((uint16_t)(v & 0xffffu))); }
__device__ __forceinline__ float hhi(uint32_t v) { return __half2float(__ushort_as_half((uint16_t)(v >> 16))); }

// acc += wa * (first texel of the pair) + wb * (second texel): FP32 weights,
// one v_fma_mix_f32 per channel and texel
__device__ __forceinline__ void acc_pair(float4 &acc, uint4 v, float wa, float wb) {
    acc.x = fmaf(hlo(v.x), wa, acc.x);
    acc.y = fmaf(hhi(v.x), wa, acc.y);
    acc.z = fmaf(hlo(v.y), wa, acc.z);
    acc.w = fmaf(hhi(v.y), wa, acc.w);
    acc.x = fmaf(hlo(v.z), wb, acc.x);
    acc.y = fmaf(hhi(v.z), wb, acc.y);
    acc.z = fmaf(hlo(v.w), wb, acc.z);
    acc.w = fmaf(hhi(v.w), wb, acc.w);
}
__device__ __forceinline__ void acc_f4(float4 &acc, uint4 v, float w) {
    acc.x = fmaf(__uint_as_float(v.x), w, acc.x);
    acc.y = fmaf(__uint_as_float(v.y), w, acc.y);
    acc.z = fmaf(__uint_as_float(v.z), w, acc.z);
    acc.w = fmaf(__uint_as_float(v.w), w, acc.w);
}
__device__ __forceinline__ void acc_face(float4 &acc, const float4 &t, float d2) {
    acc.x = fmaf(t.x, d2, acc.x);
    acc.y = fmaf(t.y, d2, acc.y);
    acc.z = fmaf(t.z, d2, acc.z);
    acc.w = fmaf(t.w, d2, acc.w);
}
// Keeps the scalar path's arithmetic out of the per-lane path's: the two end
// alike, and merged they would move every texel through vector registers.
__device__ __forceinline__ void keep_apart(float4 &acc) {
    asm volatile("" : "+v"(acc.x), "+v"(acc.y), "+v"(acc.z), "+v"(acc.w));
}

// The faces of a cone's direction: byte offsets of the three that face it, per
// lane and of the first lane, their weights dir^2, fmask (wave-uniform: bit a
// set unless weight a is 0 in every lane) and whether every lane has the first
// lane's faces.
struct ConeFaces {
    uint32_t fe[3], sfe[3];
    float d2[3];
    uint32_t fmask;
    bool fsame;
};

// The element offsets of texels i and i + 1 along an axis (i shifted by the
// border brick): the next one in the brick, or the first of the next brick.
// Brick index < 2^8, stride < 2^24 (dim <= 512): full-rate 24-bit multiplies.
__device__ __forceinline__ void axis_terms(uint32_t i, uint32_t mul, uint32_t sub, uint32_t t[2]) {
    t[0] = __umul24(i >> 2, mul) + (i & 3u) * sub;
    t[1] = t[0] + ((i & 3u) == 3u ? mul - 3u * sub : sub);
}

// The same of a wave-uniform index on the scalar unit, which has no 24-bit
// multiply (__umul24 would move the address, and the loads, to the vector side).
__device__ __forceinline__ void axis_terms_s(uint32_t i, uint32_t mul, uint32_t sub, uint32_t t[2]) {
    t[0] = (i >> 2) * mul + (i & 3u) * sub;
    t[1] = t[0] + ((i & 3u) == 3u ? mul - 3u * sub : sub);
}

// acc += lw * (trilinear sample of level l at p): isotropic, or the
// dir^2-weighted mix of the three faces that face the cone.  l is wave-uniform.
// The border bricks hold texels -1 and s as zeros, so no index is clamped and
// no weight masked; indices are shifted by one brick (+4).  What that rests on: p is
// in [0, 1] up to a few roundings.  A march leaves the box before it samples; a warped
// position is a convex mix of the warp texture's unorm16 texels, and 1 + 2^-20 still
// floors to texel s - 1 of 512.  So a shifted index is in 3 .. s + 3 and its upper
// neighbour at most s + 4, the first texel of the border brick; both are below 2^10.
// A position that is not a number passes the march's comparisons: the conversion to
// int (v_cvt_i32_f32) makes 0 of it, index 4.  Returns
// (wave-uniform) whether every texel fetched, in every lane, was +0 (ZQ: also
// test the per-lane fetches, which costs vector instructions).  An fp8 level
// reports false: its codes underflow, so a zero there does not say that the
// finer level is zero.
//
// At 1080p a wavefront's 8x8 pixels span about a voxel, so at the coarser
// levels all its lanes usually need the same 2x2x2 texels (and faces).  They
// are then fetched once for the wavefront with scalar loads and every lane
// weights them itself: the same operations on the same values as the per-lane
// path, without its vector memory traffic.  Whether they do is decided on the
// packed cell indices, before any address exists: the addresses of a shared
// cell are scalar arithmetic, and its weights are formed only if one of the
// cell's texels is not zero.  What bounds the trace is VALU issue: an empty shared cell costs 12 vector instructions (60 when
// addresses and weights were formed first), an occupied one 32 plus 36 a face.
// Texels are weighted and summed in one fixed order: a march compares its
// opacity with 0.95, and sums that differ in the last bit end some cones a step
// apart.
template <int MODE, bool ZQ>
__device__ __forceinline__ bool level_sample(float4 &acc, const PyrArgs &pa, __amdgpu_buffer_rsrc_t rs, int l,
                                             const float p[3], float lw, const ConeFaces &cf) {
    const SampleLevel &L = pa.lv[l];
    const bool aniso = L.nfaces == 6;
    const bool one = MODE == 1 || (MODE == 2 && L.one);
    const bool zq = MODE == 1 ? ZQ : (MODE == 2 && L.one ? false : ZQ);  // may a zero be reported
    float f[3];
    uint32_t i[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float u = p[k] * L.fs - 0.5f;
        const float fl = __builtin_floorf(u);
        i[k] = (uint32_t)((int)fl + 4);
        f[k] = u - fl;
    }
    const uint32_t key = i[0] | (i[1] << 10) | (i[2] << 20);
    const uint32_t k0 = __builtin_amdgcn_readfirstlane(key);
    if ((!aniso | cf.fsame) & (__ballot(key != k0) == 0)) {
        uint32_t tx[2], ty[2], tz[2], so[4];
        axis_terms_s(k0 & 1023u, L.sx, 1u, tx);
        axis_terms_s((k0 >> 10) & 1023u, L.sy, 4u, ty);
        axis_terms_s(k0 >> 20, L.sz, 16u, tz);
#pragma unroll
        for (int c = 0; c < 4; ++c) so[c] = L.org + (tx[0] + ty[c & 1] + tz[c >> 1]) * 16u;
        if (one) {
            const uint32_t dx = (tx[1] - tx[0]) * 16u;
            bool z = true;
            float w[8];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (aniso ? !((cf.fmask >> a) & 1u) : a > 0) continue;
                const uint32_t fo = aniso ? cf.sfe[a] : 0u;
                uint4 v[8];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[2 * c] = sload16(pa.pyr, so[c] + fo);
                    v[2 * c + 1] = sload16(pa.pyr, so[c] + dx + fo);
                }
                if (zero16(v)) continue;
                if (z) {
                    const float wy[2] = {1.0f - f[1], f[1]}, wz[2] = {(1.0f - f[2]) * lw, f[2] * lw};
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        w[2 * c] = ((1.0f - f[0]) * wy[c & 1]) * wz[c >> 1];
                        w[2 * c + 1] = (f[0] * wy[c & 1]) * wz[c >> 1];
                    }
                    z = false;
                }
                const float fw = aniso ? cf.d2[a] : 1.0f;
#pragma unroll
                for (int k = 0; k < 8; ++k) acc_f4(acc, v[k], w[k] * fw);
            }
            keep_apart(acc);
            return z && (MODE == 1 || !L.one);
        }
        bool z = true;
        float wa[4], wb[4];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (aniso ? !((cf.fmask >> a) & 1u) : a > 0) continue;
            uint4 v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = sload16(pa.pyr, so[c] + (aniso ? cf.sfe[a] : 0u));
            const uint64_t e0 = or16(v[0]), e1 = or16(v[1]), e2 = or16(v[2]), e3 = or16(v[3]);
            if (((e0 | e1) | (e2 | e3)) == 0) continue;
            if (z) {
                const float wy[2] = {1.0f - f[1], f[1]}, wz[2] = {(1.0f - f[2]) * lw, f[2] * lw};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float wyz = wy[c & 1] * wz[c >> 1];
                    wa[c] = (1.0f - f[0]) * wyz;
                    wb[c] = f[0] * wyz;
                }
                z = false;
            }
            float4 t = aniso ? make_float4(0.f, 0.f, 0.f, 0.f) : acc;
            if (e0) acc_pair(t, v[0], wa[0], wb[0]);
            if (e1) acc_pair(t, v[1], wa[1], wb[1]);
            if (e2) acc_pair(t, v[2], wa[2], wb[2]);
            if (e3) acc_pair(t, v[3], wa[3], wb[3]);
            if (!aniso) {
                acc = t;
                break;
            }
            acc_face(acc, t, cf.d2[a]);
        }
        keep_apart(acc);
        return z;
    }
    uint32_t tx[2], ty[2], tz[2], off[4];
    axis_terms(i[0], L.sx, 1u, tx);
    axis_terms(i[1], L.sy, 4u, ty);
    axis_terms(i[2], L.sz, 16u, tz);
#pragma unroll
    for (int c = 0; c < 4; ++c) off[c] = L.org + (tx[0] + ty[c & 1] + tz[c >> 1]) * 16u;
    const float wy[2] = {1.0f - f[1], f[1]}, wz[2] = {(1.0f - f[2]) * lw, f[2] * lw};
    bool z = zq;
    if (one) {
        const uint32_t dx = (tx[1] - tx[0]) * 16u;
        float w[8];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            w[2 * c] = ((1.0f - f[0]) * wy[c & 1]) * wz[c >> 1];
            w[2 * c + 1] = (f[0] * wy[c & 1]) * wz[c >> 1];
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (aniso ? !((cf.fmask >> a) & 1u) : a > 0) continue;
            const uint32_t fo = aniso ? cf.fe[a] : 0u;
            uint4 v[8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v[2 * c] = bload16(rs, off[c] + fo);
                v[2 * c + 1] = bload16(rs, off[c] + dx + fo);
            }
            if (zq && __ballot(!zero16(v)) == 0) continue;
            z = false;
            const float fw = aniso ? cf.d2[a] : 1.0f;
#pragma unroll
            for (int k = 0; k < 8; ++k) acc_f4(acc, v[k], w[k] * fw);
        }
        return z;
    }
    float wa[4], wb[4];
    {
        const float wlo = 1.0f - f[0], whi = f[0];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float wyz = wy[c & 1] * wz[c >> 1];
            wa[c] = wlo * wyz;
            wb[c] = whi * wyz;
        }
    }
    if (!aniso) {
        uint4 v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = bload16(rs, off[c]);
        if (zq && __ballot(!zero16(v)) == 0) return true;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc_pair(acc, v[c], wa[c], wb[c]);
        return false;
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (!((cf.fmask >> a) & 1u)) continue;
        uint4 v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = bload16(rs, off[c] + cf.fe[a]);
        if (zq && __ballot(!zero16(v)) == 0) continue;
        z = false;
        float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc_pair(t, v[c], wa[c], wb[c]);
        acc_face(acc, t, cf.d2[a]);
    }
    return z;
}

// textureLod with LINEAR_MIPMAP_LINEAR, the lambda clamp to [0, q] and the
// NEAREST magnification filter, for one wave-uniform level class D:
//   D = -1       lambda <= 0: NEAREST on level 0;
//   0 <= D < q   levels D and D+1 with weights (1 - fr, fr);
//   D = q        lambda >= q (or NaN): level q alone.
__device__ __forceinline__ int level_class(float lambda, int q, float *fr) {
    if (lambda <= 0.0f) {
        *fr = 0.0f;
        return -1;
    }
    if (!(lambda < (float)q)) {
        *fr = 0.0f;
        return q;
    }
    const float fl = __builtin_floorf(lambda);
    int d1 = (int)fl;
    d1 = d1 < 0 ? 0 : (d1 > q - 1 ? q - 1 : d1);
    *fr = lambda - fl;
    return d1;
}

template <int MODE>
__device__ __forceinline__ float4 sample_class(const PyrArgs &pa, __amdgpu_buffer_rsrc_t rs, int D, float fr,
                                               const float p[3], const ConeFaces &cf) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    const int q = pa.nlevels - 1;
    if (D < 0) {
        const int dim = pa.dim;
        const int x = (int)__builtin_floorf(p[0] * (float)dim), y = (int)__builtin_floorf(p[1] * (float)dim),
                  z = (int)__builtin_floorf(p[2] * (float)dim);
        if ((unsigned)x >= (unsigned)dim || (unsigned)y >= (unsigned)dim || (unsigned)z >= (unsigned)dim) return acc;
        const SampleLevel &L = pa.lv[0];
        uint32_t tx[2], ty[2], tz[2];
        axis_terms((uint32_t)x + 4u, L.sx, 1u, tx);
        axis_terms((uint32_t)y + 4u, L.sy, 4u, ty);
        axis_terms((uint32_t)z + 4u, L.sz, 16u, tz);
        const uint4 v = bload16(rs, L.org + (tx[0] + ty[0] + tz[0]) * 16u);
        if (MODE == 1) return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                                          __uint_as_float(v.w));
        return unpack_h4(v.x, v.y);
    }
    if (D >= q) {
        level_sample<MODE, false>(acc, pa, rs, q, p, 1.0f, cf);
        return acc;
    }
    // The coarser level first.  Its 2x2x2 cell covers the finer level's cell
    // (texels j, j+1 filter texels 2j .. 2j+3, and the finer cell around the
    // same point lies in that range), and in a nested pyramid a filtered texel
    // is zero only where every texel it filters is.  So where the coarser
    // fetch was all zero in every lane, the finer sample adds exactly 0 and is
    // skipped: cones marching through empty space.
    const bool z = level_sample<MODE, true>(acc, pa, rs, D + 1, p, fr, cf);
    if (!(z && pa.nested)) level_sample<MODE, false>(acc, pa, rs, D, p, 1.0f - fr, cf);
    return acc;
}

// traceCone (phong.frag:135-180).  ULOD: every lane of the wavefront traces a
// cone of the same aperture and initial height, so the step schedule h_i (and
// with it the sampled level) depends only on the step index and the level
// class is read from the first active lane -- or, with `sched` (the diffuse
// cones, whose schedule the host computed for the launch), read from the
// kernel arguments.  Otherwise the lanes' level classes are visited one at a
// time (each pass with a uniform class).
// WARP: warpTexture (phong.frag:150-152), each sample position goes through the
// warp texture before the pyramid is sampled (the level stays the unwarped
// one); a template argument, since the registers it takes would cost the
// unwarped tracer a wavefront per SIMD.
template <int MODE, bool ANISO, bool ULOD, bool WARP>
__device__ float4 trace_cone(const PyrArgs &pa, __amdgpu_buffer_rsrc_t rs, const float pos[3], const float nrm[3],
                             const float dir_in[3], int steps, float bias, float tan_half, float h0,
                             float lod_offset, const float4 *warp, const ConeSchedule *sched = nullptr) {
    float dir[3];
    {
        const float il = __builtin_amdgcn_rsqf(dot3(dir_in, dir_in));
        dir[0] = dir_in[0] * il;
        dir[1] = dir_in[1] * il;
        dir[2] = dir_in[2] * il;
    }
    ConeFaces cf = {{0u, 0u, 0u}, {0u, 0u, 0u}, {0.f, 0.f, 0.f}, 0u, true};
    if (ANISO) {
        uint32_t fk = 0u;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t face = (uint32_t)(2 * k + (dir[k] >= 0.0f ? 0 : 1));
            cf.fe[k] = 1024u * face;
            cf.sfe[k] = __builtin_amdgcn_readfirstlane(cf.fe[k]);
            cf.d2[k] = dir[k] * dir[k];
            // cones along a grid axis (faces of axis-aligned walls) weight only
            // one or two of the three faces
            if (__ballot(cf.d2[k] != 0.0f) != 0) cf.fmask |= 1u << k;
            fk |= face << (4 * k);
        }
        cf.fsame = __ballot(__builtin_amdgcn_readfirstlane(fk) != fk) == 0;
    }
    const int q = pa.nlevels - 1;
    float c0 = 0.f, c1 = 0.f, c2 = 0.f, a = 0.f;
    const float scale = 1.0f / (float)pa.dim;
    float start[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) start[k] = pos[k] + (bias * nrm[k]) * scale;
    if (ULOD && sched != nullptr && sched->n == steps) {
        // dim is a power of two, so (h * dir) * scale == h * (dir * scale) exactly
        float ds[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) ds[k] = dir[k] * scale;
        for (int i = 0; i < steps && a < 0.95f; ++i) {
            const float h = sched->h[i];
            float sp[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) sp[k] = start[k] + h * ds[k];
            if (fminf(fminf(sp[0], sp[1]), sp[2]) < 0.f || fmaxf(fmaxf(sp[0], sp[1]), sp[2]) > 1.f) break;
            if (WARP) warp_sample_march(warp, sp);
            const float4 smp = sample_class<MODE>(pa, rs, sched->cls[i], sched->fr[i], sp, cf);
            const float aa = 1.0f - a;
            c0 += smp.x * aa;
            c1 += smp.y * aa;
            c2 += smp.z * aa;
            a += aa * smp.w;
        }
        return make_float4(c0, c1, c2, a);
    }
    float h = h0;
    for (int i = 0; i < steps && a < 0.95f; ++i) {
        const float r = h * tan_half;
        const float lod = __builtin_amdgcn_logf(fmaxf(1.0f, 2.0f * r));  // v_log_f32: argument >= 1, no denormals
        float sp[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) sp[k] = start[k] + (h * dir[k]) * scale;
        if (fminf(fminf(sp[0], sp[1]), sp[2]) < 0.f || fmaxf(fmaxf(sp[0], sp[1]), sp[2]) > 1.f) break;
        if (WARP) warp_sample_march(warp, sp);
        float fr;
        const int D = level_class(lod + lod_offset, q, &fr);
        float4 smp;
        if (ULOD) {
            const int Du = __builtin_amdgcn_readfirstlane(D);
            const float fru = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fr)));
            smp = sample_class<MODE>(pa, rs, Du, fru, sp, cf);
        } else {
            smp = make_float4(0.f, 0.f, 0.f, 0.f);
            bool pending = true;
            while (true) {
                const uint64_t m = __ballot(pending);
                if (m == 0) break;
                const int Du = __builtin_amdgcn_readlane(D, __builtin_ctzll(m));
                if (pending && D == Du) {
                    smp = sample_class<MODE>(pa, rs, Du, fr, sp, cf);
                    pending = false;
                }
            }
        }
        const float aa = 1.0f - a;
        c0 += smp.x * aa;
        c1 += smp.y * aa;
        c2 += smp.z * aa;
        a += aa * smp.w;
        h += r;
    }
    return make_float4(c0, c1, c2, a);
}

static __constant__ float kConeDirs[6][3] = {{0.0f, 1.0f, 0.0f},
                                      {0.0f, 0.5f, 0.866025f},
                                      {0.823639f, 0.5f, 0.267617f},
                                      {0.509037f, 0.5f, -0.700629f},
                                      {-0.5909037f, 0.5f, -0.700629f},  // sic: phong.frag:475
                                      {-0.823639f, 0.5f, 0.267617f}};
static __constant__ float kConeW[6] = {0.25f, 0.15f, 0.15f, 0.15f, 0.15f, 0.15f};

// A G-buffer texel as the gather uses it: texture-space position, unit normal,
// tangent frame.
struct TracePixel {
    float gp[3], pos[3], N[3], nraw[3], T[3], B[3], rough;
    bool covered;
};
__device__ __forceinline__ void load_pixel(const TraceLaunch &t, size_t pi, TracePixel &x) {
    const float4 *g = (const float4 *)&t.gbuf[pi];
    const float4 g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
    x.covered = __float_as_uint(g2.w) != 0u;
    x.gp[0] = g0.x;
    x.gp[1] = g0.y;
    x.gp[2] = g0.z;
#pragma unroll
    for (int k = 0; k < 3; ++k) x.pos[k] = ((x.gp[k] - t.ext.center[k]) - t.ext.vmin[k]) / (t.ext.vmax[k] - t.ext.vmin[k]);
    x.nraw[0] = g1.x;
    x.nraw[1] = g1.y;
    x.nraw[2] = g1.z;
    x.rough = g1.w;
    x.T[0] = g2.x;
    x.T[1] = g2.y;
    x.T[2] = g2.z;
    x.B[0] = g3.x;
    x.B[1] = g3.y;
    x.B[2] = g3.z;
    nrm3(x.nraw, x.N);
}

// Diffuse cone i of the gather (phong.frag:480-484).
template <int MODE, bool ANISO, bool WARP>
__device__ __forceinline__ float4 diffuse_cone(const TraceLaunch &t, const PyrArgs &pa, __amdgpu_buffer_rsrc_t rs,
                                               const TracePixel &x, int i) {
    const float cx = kConeDirs[i][0], cy = kConeDirs[i][1], cz = kConeDirs[i][2];
    float d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k] = (x.T[k] * cx + x.B[k] * cy) + x.nraw[k] * cz;
    return trace_cone<MODE, ANISO, true, WARP>(pa, rs, x.pos, x.N, d, t.d_steps, t.d_bias, t.d_tan_half, t.d_h0,
                                               t.d_lod_offset, t.warp, &t.d_sched);
}

// The weighted sum of the diffuse cones, one cone at a time in order, and its
// image value (phong.frag:483-489).
__device__ __forceinline__ void add_cone(float4 &sum, const float4 &r, int i) {
    const float w = kConeW[i];
    sum.x += w * r.x;
    sum.y += w * r.y;
    sum.z += w * r.z;
    sum.w += w * r.w;
}
__device__ __forceinline__ float4 indirect_value(const TraceLaunch &t, const float4 &sum) {
    const float occ = 1.0f - clampf(sum.w, 0.0f, 1.0f);
    const float m = t.draw_occlusion ? occ : 1.0f;
    return make_float4(sum.x * m, sum.y * m, sum.z * m, occ);
}

// The specular cone (phong.frag:491-512).
template <int MODE, bool ANISO, bool WARP>
__device__ __forceinline__ float4 specular_cone(const TraceLaunch &t, const PyrArgs &pa, __amdgpu_buffer_rsrc_t rs,
                                                const TracePixel &x) {
    float angle = t.s_angle;
    if (t.angle_from_roughness && t.has_roughness) angle = (x.rough * 3.1415982f) * 0.1f;  // PI of common.glsl:1
    const float I[3] = {x.gp[0] - t.eye[0], x.gp[1] - t.eye[1], x.gp[2] - t.eye[2]};
    const float dni = dot3(x.N, I);
    float R[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) R[k] = I[k] - (2.0f * dni) * x.N[k];
    const float th = tanf(angle / 2.0f);
    // One material under the whole wavefront (the usual case): every lane's
    // cone has the same aperture, so the step schedule and the level classes
    // are the same in every lane.
    const float th0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(th)));
    if (__ballot(__float_as_int(th) != __float_as_int(th0)) == 0)
        return trace_cone<MODE, ANISO, true, WARP>(pa, rs, x.pos, x.N, R, t.s_steps, t.s_bias, th, t.s_h0,
                                                   t.s_lod_offset, t.warp);
    return trace_cone<MODE, ANISO, false, WARP>(pa, rs, x.pos, x.N, R, t.s_steps, t.s_bias, th, t.s_h0, t.s_lod_offset,
                                                t.warp);
}

inline PyrArgs pyr_args(const PyrDesc &pyr, int nested) {
    PyrArgs a;
    a.pyr = pyr.pyr;
    a.bytes = pyr.bytes;
    a.dim = pyr.dim;
    a.nlevels = pyr.nlevels;
    a.nested = nested;
    for (int l = 0; l < VCT_MAX_LEVELS; ++l) {
        const LevelInfo &L = pyr.lv[l < pyr.nlevels ? l : 0];
        a.lv[l] = SampleLevel{(float)L.size, L.stage - L.pad * 16u, L.sx, L.sy, L.sz, L.nfaces, L.fmt != 0 ? 1 : 0, 0};
    }
    return a;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pyr_rsrc(const PyrArgs &pa) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)pa.pyr, (short)0, (int)pa.bytes, 0x00020000);
}

}  // namespace vctk
