// scan.hip -- item offsets for the binned rasterizer, chunk starts, fills.
#include "vct_device.h"

namespace vctk {

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(256) void k_reduce_stats(const uint32_t *partials, int n, uint32_t *sum0, uint32_t *max1,
                                                      uint32_t *sum2) {
    uint32_t a = 0, b = 0, c = 0;
    for (int i = threadIdx.x; i < n; i += 256) {
        a += partials[i * 4 + 0];
        b = partials[i * 4 + 1] > b ? partials[i * 4 + 1] : b;
        c += partials[i * 4 + 2];
    }
    __shared__ uint32_t red[3][256];
    red[0][threadIdx.x] = a;
    red[1][threadIdx.x] = b;
    red[2][threadIdx.x] = c;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] = red[1][threadIdx.x + s] > red[1][threadIdx.x] ? red[1][threadIdx.x + s] : red[1][threadIdx.x];
            red[2][threadIdx.x] += red[2][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (sum0) *sum0 = red[0][0];
        if (max1) *max1 = red[1][0];
        if (sum2) *sum2 = red[2][0];
    }
}

hipError_t launch_reduce_stats(const uint32_t *partials, int n, uint32_t *sum0, uint32_t *max1, uint32_t *sum2,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_reduce_stats, dim3(1), dim3(256), 0, s, partials, n, sum0, max1, sum2);
    return hipGetLastError();
}

static unsigned fill_blocks(size_t n) {
    size_t b = (n + 255) / 256;
    return (unsigned)(b > 4096 ? 4096 : (b == 0 ? 1 : b));
}

hipError_t launch_fill_u32(uint32_t *p, uint32_t v, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u32, dim3(fill_blocks(n)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- raster scan
// The item offsets of the binned rasterizer: counts[0..n) (and, for the passes
// with a block walk, bcounts[0..n)) -> exclusive offsets offs[0..n] (offs[n] =
// total) and the chunk starts chunk[c] = the slot holding item 64 c, for both
// arrays together, a workgroup per tile of 2048 slots.  What is in front of a
// tile is added up by the tile's own workgroup: up to kScanDirect tiles from the
// counts (one launch), up to kScanWide from the tiles' sums (a launch before),
// and beyond that, where the sums of all tiles for every tile are more than the
// slots themselves, one workgroup turns the sums into prefixes first.
//
// What bounds it: latency, then the 24 bytes per slot.  It was always the three
// launches, with the chunk starts written slot by slot (a wavefront waited for
// its widest slots).  A single launch that passes prefixes from tile to tile
// took longer than all three: the words cross the XCDs (28 us for 23 at 0.1 to
// 0.6 million slots).  A frame's three scans: 36 triangles 48 us before, 18; 0.35
// million triangles with 5 lights 69 us, 51, and 138 us, 59 with the 512^3 grid's
// wide slots (two scans); 21.7 million slots of 8 lights 200 us, 204 (its bytes).
constexpr int kScanThreads = 256, kScanPer = 8, kScanTile = kScanThreads * kScanPer;
// tiles: with 8 the last one reads the 7 in front of it (6 us in one launch; sums
// and offsets 10); with 2048 it reads 32 KB of sums (at 10,600 all of them 0.9 GB)
constexpr int kScanDirect = 8, kScanWide = 2048;

size_t raster_scan_tiles(size_t nslots) { return (nslots + kScanTile - 1) / kScanTile; }

__device__ __forceinline__ void scan_load8(const uint32_t *__restrict__ a, size_t n, size_t base, uint32_t v[8]) {
    if (base + 8 <= n) {
        const uint4 x = *(const uint4 *)(a + base), y = *(const uint4 *)(a + base + 4);
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = base + j < n ? a[base + j] : 0u;
    }
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t x) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
    return x;
}

// inclusive prefix sum over the lanes of a wavefront
__device__ __forceinline__ uint64_t wave_incl_u64(uint64_t x, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    return x;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_tile_sums(const uint32_t *__restrict__ a,
                                                                 const uint32_t *__restrict__ b, size_t n,
                                                                 uint64_t *tsum) {
    __shared__ uint64_t red[2][kScanThreads / 64];
    const size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanPer;
    uint32_t v[8];
    uint64_t sa = 0, sb = 0;
    scan_load8(a, n, base, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) sa += v[j];
    if (b) {
        scan_load8(b, n, base, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) sb += v[j];
    }
    sa = wave_sum_u64(sa);
    sb = wave_sum_u64(sb);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[0][w] = sa;
        red[1][w] = sb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t ta = 0, tb = 0;
        for (int i = 0; i < kScanThreads / 64; ++i) {
            ta += red[0][i];
            tb += red[1][i];
        }
        tsum[2 * blockIdx.x] = ta;
        tsum[2 * blockIdx.x + 1] = tb;
    }
}

// One workgroup: exclusive prefixes of the tile sums (both arrays) and the
// totals offs[n], boffs[n].
__global__ __launch_bounds__(1024) void k_scan_tiles(const uint64_t *__restrict__ tsum, int ntiles, uint64_t *tpre,
                                                     uint64_t *end_a, uint64_t *end_b) {
    __shared__ uint64_t wt[2][16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int per = (ntiles + 1023) / 1024;
    const int t0 = t * per, t1 = t0 + per < ntiles ? t0 + per : ntiles;
    uint64_t sa = 0, sb = 0;
    for (int i = t0; i < t1; ++i) {
        sa += tsum[2 * i];
        sb += tsum[2 * i + 1];
    }
    const uint64_t ia = wave_incl_u64(sa, lane), ib = wave_incl_u64(sb, lane);
    if (lane == 63) {
        wt[0][w] = ia;
        wt[1][w] = ib;
    }
    __syncthreads();
    uint64_t pa = ia - sa, pb = ib - sb, ta = 0, tb = 0;
    for (int i = 0; i < 16; ++i) {
        if (i < w) {
            pa += wt[0][i];
            pb += wt[1][i];
        }
        ta += wt[0][i];
        tb += wt[1][i];
    }
    for (int i = t0; i < t1; ++i) {
        tpre[2 * i] = pa;
        tpre[2 * i + 1] = pb;
        pa += tsum[2 * i];
        pb += tsum[2 * i + 1];
    }
    if (t == 0) {
        *end_a = ta;
        if (end_b) *end_b = tb;
    }
}

struct ScanLds {
    uint32_t mark[kScanTile];
    uint32_t last[kScanThreads / 64];
};

// One array's offsets and chunk starts of the tile at slot t0, whose items are
// [start, end); p is this thread's exclusive prefix.  The chunks of the tile
// are written kScanTile at a time: every slot marks the first chunk that starts
// in it (no two mark the same), and a running maximum over the marks gives
// every chunk its slot.
__device__ __forceinline__ void scan_write(const uint32_t v[8], size_t n, size_t t0, uint64_t p, uint64_t start,
                                           uint64_t end, uint64_t *offs, uint32_t *chunk, size_t cap, ScanLds &lds) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t base = t0 + (size_t)threadIdx.x * kScanPer;
    uint64_t o[9];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        o[j] = p;
        p += v[j];
    }
    o[8] = p;
    if (base + 8 <= n) {
        ulonglong2 *d = (ulonglong2 *)(offs + base);
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = make_ulonglong2(o[2 * j], o[2 * j + 1]);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (base + j < n) offs[base + j] = o[j];
    }
    const uint64_t c0 = (start + 63) >> 6, c1 = (end + 63) >> 6 < cap ? (end + 63) >> 6 : cap;
    uint32_t carry = 0;  // 1 + the slot of the last chunk in front of these
    for (uint64_t cw = c0 & ~(uint64_t)7; cw < c1; cw += kScanTile) {
        uint4 *mine = (uint4 *)(lds.mark + threadIdx.x * kScanPer);
        __syncthreads();  // the marks before these have been read
        mine[0] = mine[1] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint64_t s = (o[j] + 63) >> 6, e = (o[j + 1] + 63) >> 6;
            if (s < e && s - cw < (uint64_t)kScanTile) lds.mark[s - cw] = threadIdx.x * kScanPer + j + 1;
        }
        __syncthreads();
        const uint4 x = mine[0], y = mine[1];
        uint32_t m[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
        for (int j = 1; j < 8; ++j) m[j] = m[j] > m[j - 1] ? m[j] : m[j - 1];
        uint32_t top = m[7];  // -> the lanes' running maximum
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t z = __shfl_up(top, d, 64);
            if (lane >= d && z > top) top = z;
        }
        if (lane == 63) lds.last[w] = top;
        uint32_t front = __shfl_up(top, 1, 64);
        if (lane == 0) front = 0;
        __syncthreads();
        front = front > carry ? front : carry;
#pragma unroll
        for (int i = 0; i < kScanThreads / 64; ++i) {
            const uint32_t z = lds.last[i];
            if (i < w && z > front) front = z;
            if (z > carry) carry = z;
        }
        const uint32_t t1 = (uint32_t)t0 - 1;
#pragma unroll
        for (int j = 0; j < 8; ++j) m[j] = (m[j] > front ? m[j] : front) + t1;
        const uint64_t c = cw + threadIdx.x * kScanPer;
        if (c >= c0 && c + 8 <= c1) {
            ((uint4 *)(chunk + c))[0] = make_uint4(m[0], m[1], m[2], m[3]);
            ((uint4 *)(chunk + c))[1] = make_uint4(m[4], m[5], m[6], m[7]);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (c + j >= c0 && c + j < c1) chunk[c + j] = m[j];
        }
    }
}

// before: the tiles' prefixes (PREFIX), their sums, or null (from the counts).
template <bool PREFIX>
__global__ __launch_bounds__(kScanThreads) void k_scan_offsets(const uint32_t *__restrict__ a,
                                                               const uint32_t *__restrict__ b, size_t n,
                                                               const uint64_t *__restrict__ before, uint64_t *offs_a,
                                                               uint64_t *offs_b, uint32_t *chunk_a, uint32_t *chunk_b,
                                                               size_t cap) {
    __shared__ uint64_t wt[4][kScanThreads / 64];
    __shared__ ScanLds lds;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, tile = blockIdx.x;
    const size_t t0 = (size_t)tile * kScanTile, base = t0 + (size_t)threadIdx.x * kScanPer;
    uint32_t va[8], vb[8] = {};
    uint64_t sa = 0, sb = 0, fa = 0, fb = 0;  // the tile's, and the tiles' in front of it
    scan_load8(a, n, base, va);
    if (b) scan_load8(b, n, base, vb);
    if (!PREFIX && before) {
        for (int i = threadIdx.x; i < tile; i += kScanThreads) {
            const ulonglong2 x = ((const ulonglong2 *)before)[i];
            fa += x.x;
            fb += x.y;
        }
    } else if (!PREFIX) {
        for (size_t i = threadIdx.x; i < t0 / 4; i += kScanThreads) {  // whole tiles: no remainder
            const uint4 x = ((const uint4 *)a)[i];
            fa += ((uint64_t)x.x + x.y) + ((uint64_t)x.z + x.w);
            if (b) {
                const uint4 y = ((const uint4 *)b)[i];
                fb += ((uint64_t)y.x + y.y) + ((uint64_t)y.z + y.w);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        sa += va[j];
        sb += vb[j];
    }
    const uint64_t ia = wave_incl_u64(sa, lane), ib = b ? wave_incl_u64(sb, lane) : 0;
    if (!PREFIX && tile > 0) {
        fa = wave_sum_u64(fa);
        if (b) fb = wave_sum_u64(fb);
    }
    if (lane == 63) {
        wt[0][w] = ia;
        wt[1][w] = ib;
        wt[2][w] = fa;
        wt[3][w] = fb;
    }
    __syncthreads();
    uint64_t pa = ia - sa, pb = ib - sb, ta = 0, tb = 0;
    fa = PREFIX ? before[2 * tile] : 0;
    fb = PREFIX ? before[2 * tile + 1] : 0;
#pragma unroll
    for (int i = 0; i < kScanThreads / 64; ++i) {
        if (i < w) {
            pa += wt[0][i];
            pb += wt[1][i];
        }
        ta += wt[0][i];
        tb += wt[1][i];
        if (!PREFIX) {
            fa += wt[2][i];
            fb += wt[3][i];
        }
    }
    scan_write(va, n, t0, fa + pa, fa, fa + ta, offs_a, chunk_a, cap, lds);
    if (b) scan_write(vb, n, t0, fb + pb, fb, fb + tb, offs_b, chunk_b, cap, lds);
    if (!PREFIX && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        offs_a[n] = fa + ta;
        if (b) offs_b[n] = fb + tb;
    }
}

hipError_t raster_scan(RasterScratch &rs, size_t nslots, bool blocks, hipStream_t s) {
    const size_t ntiles = raster_scan_tiles(nslots);
    if (ntiles > rs.scan_tiles_cap || ntiles == 0) return hipErrorInvalidValue;
    const uint32_t *b = blocks ? rs.bcounts : nullptr;
    uint64_t *const pre = rs.tsum + 2 * rs.scan_tiles_cap;
    const dim3 grid((unsigned)ntiles), block(kScanThreads);
    hipError_t e;
    if (ntiles > (size_t)kScanDirect) {
        hipLaunchKernelGGL(k_scan_tile_sums, grid, block, 0, s, rs.counts, b, nslots, rs.tsum);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (ntiles > (size_t)kScanWide) {
        hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(1024), 0, s, rs.tsum, (int)ntiles, pre, rs.offs + nslots,
                           blocks ? rs.boffs + nslots : nullptr);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(k_scan_offsets<true>, grid, block, 0, s, rs.counts, b, nslots, pre, rs.offs, rs.boffs,
                           rs.chunk, rs.bchunk, rs.chunk_cap);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_scan_offsets<false>, grid, block, 0, s, rs.counts, b, nslots,
                       ntiles > (size_t)kScanDirect ? rs.tsum : nullptr, rs.offs, rs.boffs, rs.chunk, rs.bchunk,
                       rs.chunk_cap);
    return hipGetLastError();
}

}  // namespace vctk
