// sl_geom.hip -- scans, vertex transform/cull, monotone split + fragment counting and
// curve / cut-line intersection (the "ts" array) of the comb-scanline pipeline.
#include "sl_device.h"
#include "sl_internal.h"

#include <algorithm>

namespace sl {
using namespace dev;

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}

// Exclusive scan of the 256 per-thread values of a block; returns the block total.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t &total, uint32_t *lds /*[4]*/) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) lds[wid] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        uint32_t x = lds[w];
        if (w < wid) off += x;
        tot += x;
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

// What a scan reads: up to two arrays in one launch (blockIdx.y), or the bucket count of every
// path, worked out from its row range.
struct ScanArrays {
    const uint32_t *in[2];
    __device__ __forceinline__ uint32_t operator()(int y, size_t i) const { return in[y][i]; }
};
struct ScanPathBuckets {
    const int2 *prow;
    __device__ __forceinline__ uint32_t operator()(int, size_t i) const { return path_bucket_count(prow[i]); }
};
struct ScanOut {
    uint32_t *out[2];
    uint32_t *tmp[2];  // tile totals
};

template <class In>
__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(In in, size_t n, ScanOut o) {
    __shared__ uint32_t lds[4];
    const int y = blockIdx.y;
    size_t base = (size_t)blockIdx.x * kScanTile;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        size_t i = base + (size_t)k * kScanThreads + threadIdx.x;
        if (i < n) s += in(y, i);
    }
    uint32_t tot;
    block_excl_scan(s, tot, lds);
    if (threadIdx.x == 0) o.tmp[y][blockIdx.x] = tot;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_top(uint32_t *tile_sum, size_t ntiles, uint32_t *out_total) {
    __shared__ uint32_t lds[4];
    uint32_t carry = 0;
    for (size_t c = 0; c < ntiles; c += kScanThreads) {
        size_t i = c + threadIdx.x;
        uint32_t v = i < ntiles ? tile_sum[i] : 0u;
        uint32_t tot;
        uint32_t ex = block_excl_scan(v, tot, lds);
        if (i < ntiles) tile_sum[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) *out_total = carry;
}

// The down-sweep.  DIRECT, for scans of at most kScanDirectTiles tiles: each block sums the
// tile totals before its own (at most 4095 L2-resident words) instead of a separate pass
// scanning them, and the last block writes the grand total to out[n].
constexpr size_t kScanDirectTiles = 4096;

template <bool DIRECT, class In>
__global__ void __launch_bounds__(kScanThreads) k_scan_down(In in, size_t n, ScanOut o) {
    __shared__ uint32_t lds[4];
    const int y = blockIdx.y;
    const uint32_t *tile = o.tmp[y];
    uint32_t *out = o.out[y];
    uint32_t tile_off = 0;
    if (DIRECT) {
        uint32_t pre = 0;
        for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kScanThreads) pre += tile[i];
        block_excl_scan(pre, tile_off, lds);
    } else {
        tile_off = tile[blockIdx.x];
    }
    size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        size_t i = base + k;
        v[k] = i < n ? in(y, i) : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t ex = block_excl_scan(s, tot, lds) + tile_off;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        size_t i = base + k;
        if (i < n) out[i] = ex;
        ex += v[k];
    }
    if (DIRECT && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = tile_off + tot;
}

// A whole scan in one launch, a block an array: up to 16 values a thread.  One launch of about
// 5 us where the two passes take 3 to 4 us each; beyond that size one block is the slower.
constexpr int kScanSmallThreads = 1024, kScanSmallItems = 16;
constexpr size_t kScanSmall = (size_t)kScanSmallThreads * kScanSmallItems;

template <class In>
__global__ void __launch_bounds__(kScanSmallThreads) k_scan_small(In in, size_t n, ScanOut o) {
    __shared__ uint32_t part[kScanSmallThreads / 64];
    const int y = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t base = (size_t)threadIdx.x * kScanSmallItems;
    uint32_t v[kScanSmallItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanSmallItems; ++k) {
        v[k] = base + k < n ? in(y, base + k) : 0u;
        s += v[k];
    }
    const uint32_t inc = wave_incl_scan(s);
    if (lane == 63) part[wv] = inc;
    __syncthreads();
    uint32_t ex = inc - s, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanSmallThreads / 64; ++w) {
        if (w < wv) ex += part[w];
        tot += part[w];
    }
    uint32_t *out = o.out[y];
#pragma unroll
    for (int k = 0; k < kScanSmallItems; ++k) {
        if (base + k < n) out[base + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0) out[n] = tot;
}

template <class In>
void scan_launch(const In &in, int arrays, const ScanOut &o, size_t n, hipStream_t s) {
    if (n <= kScanSmall) {
        hipLaunchKernelGGL(k_scan_small<In>, dim3(1, arrays), dim3(kScanSmallThreads), 0, s, in, n, o);
        return;
    }
    const size_t ntiles = (n + kScanTile - 1) / kScanTile;
    const dim3 g((unsigned)ntiles, arrays), b(kScanThreads);
    hipLaunchKernelGGL(k_scan_reduce<In>, g, b, 0, s, in, n, o);
    if (ntiles <= kScanDirectTiles) {
        hipLaunchKernelGGL((k_scan_down<true, In>), g, b, 0, s, in, n, o);
        return;
    }
    for (int y = 0; y < arrays; ++y)
        hipLaunchKernelGGL(k_scan_top, dim3(1), b, 0, s, o.tmp[y], ntiles, o.out[y] + n);
    hipLaunchKernelGGL((k_scan_down<false, In>), g, b, 0, s, in, n, o);
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_u8(uint8_t *p, uint8_t v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// rows of `row_bytes` bytes, `pitch` apart (the bytes between rows are left alone)
__global__ void k_fill_rows_u8(uint8_t *p, uint8_t v, size_t row_bytes, size_t pitch, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[(i / row_bytes) * pitch + i % row_bytes] = v;
}

inline unsigned blocks_for(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

// VALU issue-rate probe: every thread runs `iters` rounds of 64 steps of 8 independent fma
// chains, i.e. 512 v_fma_f32 per round and wave, nothing else in the loop body but the
// loop counter (scalar).  Timed over a full grid it gives the wave VALU instructions per
// second the machine issues.
__global__ void __launch_bounds__(256) k_valu_probe(int iters, float seed, float *out) {
    float a0 = seed + threadIdx.x, a1 = a0 + 1.f, a2 = a0 + 2.f, a3 = a0 + 3.f;
    float a4 = a0 + 4.f, a5 = a0 + 5.f, a6 = a0 + 6.f, a7 = a0 + 7.f;
    const float m = 0.999f, c = 1e-3f;
    for (int i = 0; i < iters; ++i) {
#pragma unroll
        for (int k = 0; k < 64; ++k) {
            a0 = __builtin_fmaf(a0, m, c); a1 = __builtin_fmaf(a1, m, c);
            a2 = __builtin_fmaf(a2, m, c); a3 = __builtin_fmaf(a3, m, c);
            a4 = __builtin_fmaf(a4, m, c); a5 = __builtin_fmaf(a5, m, c);
            a6 = __builtin_fmaf(a6, m, c); a7 = __builtin_fmaf(a7, m, c);
        }
    }
    const float r = ((a0 + a1) + (a2 + a3)) + ((a4 + a5) + (a6 + a7));
    if (r == 12345.f) out[blockIdx.x] = r;  // keeps the chains live; never true in practice
}

// ------------------------------------------------------------------------------------
// per-path init, vertex transform + region flags (k_transformVertex, .cu:36-105)
// ------------------------------------------------------------------------------------
__global__ void k_frame_init(uint32_t P, uint32_t *pflags, int2 *prow, uint32_t *small) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kFrameStatusWords) small[p] = 0u;
    if (p >= P) return;
    pflags[p] = 0u;
    prow[p] = make_int2(INT_MAX, INT_MIN);
}

// the three sizes a frame's host side needs, written to pinned host memory in one launch
__global__ void k_sizes(const uint32_t *F, const uint32_t *NCH, const uint32_t *NB, uint32_t *host) {
    if (threadIdx.x == 0) {
        host[0] = *F;
        host[1] = *NCH;
        host[2] = *NB;
        __threadfence_system();
    }
}

struct Mat4 { float m[16]; };

__global__ void k_transform(uint32_t V, const float2 *__restrict__ vtx, const uint32_t *__restrict__ vpath,
                            const int4 *__restrict__ pcanvas, Mat4 M, int W, int H, float2 *__restrict__ out,
                            uint32_t *pflags) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < V;
    const uint32_t p = live ? vpath[i] : 0u;
    if (pcanvas && live) {
        const int4 cv = pcanvas[p];
        W = cv.x;
        H = cv.y;
    }
    const float2 iv = live ? vtx[i] : make_float2(0.f, 0.f);
    const float ix = iv.x, iy = iv.y, iz = 0.f, iw = 1.f;
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        o[k] = M.m[4 * k + 0] * ix + M.m[4 * k + 1] * iy + M.m[4 * k + 2] * iz + M.m[4 * k + 3] * iw;
    if (o[3] != 1.f) {  // an affine transform's w: the quotients are the values themselves
        o[0] /= o[3];
        o[1] /= o[3];
        o[2] /= o[3];
    }
    const float w = (float)W, h = (float)H;
    const float z = (float)(W < H ? W : H);
    const float cutoff = -z * 0.5f;
    if (o[2] < cutoff) o[2] = cutoff;
    const float w2 = w * .5f, h2 = h * .5f;
    float ox = (o[0] - w2) * z / (o[2] + z) + w2;
    float oy = (o[1] - h2) * z / (o[2] + z) + h2;
    int xf = ox < 0 ? 0 : (ox <= w ? 1 : 2);
    int yf = oy < 0 ? 0 : (oy <= h ? 1 : 2);
    // region bit per the 3x3 layout of ras_define.h:104-117: regions r = 3 yf + xf take bits
    // 0, 1, 2, 3, -, 4, 5, 6, 7 in order; the inside (r = 4) sets bits 0 and 7
    const int r = 3 * yf + xf;
    const uint32_t bits = r == 4 ? ((1u << 0) | (1u << 7)) : 1u << (r - (r > 4 ? 1 : 0));
    // OR the region bits into the path's flags: one atomic per distinct path of the wave
    const int lane = threadIdx.x & 63;
    uint64_t pend = __ballot(live);
    while (pend) {
        const int leader = __ffsll((long long)pend) - 1;
        const uint32_t lp = (uint32_t)__builtin_amdgcn_readlane((int)p, leader);
        const bool mine = ((pend >> lane) & 1ull) && p == lp;
        const uint64_t grp = __ballot(mine);
        // the group's OR of the eight region bits: mostly the leader's own, else one ballot a
        // bit (scalar results, no cross-lane data movement)
        uint32_t acc = (uint32_t)__builtin_amdgcn_readlane((int)bits, leader);
        if (__ballot(mine && bits != acc)) {
#pragma unroll
            for (int b = 0; b < 8; ++b) acc |= __ballot(mine && ((bits >> b) & 1u)) ? (1u << b) : 0u;
        }
        if (lane == leader) atomicOr(&pflags[lp], acc);
        pend &= ~grp;
    }
    if (!live) return;
    if (floorf(ox) == ox) ox = ox - 1.f / 256.f;
    out[i] = make_float2(ox, oy);
}

// ------------------------------------------------------------------------------------
// curve loading
// ------------------------------------------------------------------------------------
struct Curve {
    int type;
    float w;
    float x0, x1, x2, x3, y0, y1, y2, y3;
};

// A curve and its monotone cuts from its 64-byte record (k_monotone writes it): {x0, y0, x1, y1},
// {x2, y2, x3, y3}, {cuts}, {type | cuts << 8, w, path, vertex order reversed}.  One cache line per
// curve for the intersection passes, whose work lists visit curves out of order.
struct CurveRec {
    Curve cu;
    float4 q;       // monotone cuts
    int n;          // cut count
    uint32_t path;
};

__device__ __forceinline__ CurveRec load_rec(const float4 *__restrict__ crec, uint32_t c) {
    CurveRec r;
    const float4 a = crec[4 * (size_t)c], b = crec[4 * (size_t)c + 1];
    r.q = crec[4 * (size_t)c + 2];
    const float4 m = crec[4 * (size_t)c + 3];
    const uint32_t tw = fb(m.x);
    r.cu.type = (int)(tw & 0xFFu);
    r.n = (int)((tw >> 8) & 0xFFu);
    r.cu.w = m.y;
    r.path = fb(m.z);
    r.cu.x0 = a.x; r.cu.y0 = a.y; r.cu.x1 = a.z; r.cu.y1 = a.w;
    r.cu.x2 = b.x; r.cu.y2 = b.y; r.cu.x3 = b.z; r.cu.y3 = b.w;
    return r;
}

__device__ __forceinline__ Curve load_curve(const SceneDev &sc, const float2 *__restrict__ tv, uint32_t c) {
    Curve cu;
    const uint4 ci = sc.cinfo[c];
    cu.type = (int)(ci.z & 0xFFu);
    cu.w = (cu.type == CT_RATIONAL) ? bf(ci.w) : 0.f;
    const uint32_t p = ci.x;
    const int nv = cu.type & 7;
    float2 a = tv[p], b = tv[p + 1];
    float2 d = nv > 2 ? tv[p + 2] : make_float2(0.f, 0.f);
    float2 e = nv > 3 ? tv[p + 3] : make_float2(0.f, 0.f);
    cu.x0 = a.x; cu.y0 = a.y; cu.x1 = b.x; cu.y1 = b.y;
    cu.x2 = d.x; cu.y2 = d.y; cu.x3 = e.x; cu.y3 = e.y;
    return cu;
}
__device__ __forceinline__ float ex(const Curve &c, float t) { return curve_eval(c.type, c.w, c.x0, c.x1, c.x2, c.x3, t); }
__device__ __forceinline__ float ey(const Curve &c, float t) { return curve_eval(c.type, c.w, c.y0, c.y1, c.y2, c.y3, t); }

// Monotone split points of one coordinate (k_make_intersection_0, ras_cut.h:1314-1409)
__device__ __forceinline__ void monotone_axis(const Curve &c, float v0, float v1, float v2, float v3, float *tq, int &n) {
    if (c.type == CT_QUAD) {
        float b = (v0 - v1) + (v2 - v1);
        if (!(fabsf(b) < 1e-6f)) {
            float t = (v0 - v1) / b;
            if (t > 0.f && t < 1.f) { tq[n] = t; n++; }
        }
    } else if (c.type == CT_CUBIC) {
        float r0 = 0.f, r1 = 0.f;
        solve_quad((v3 - v0) + 3.f * (v1 - v2), 2.f * ((v0 - v1) + (v2 - v1)), v1 - v0, r0, r1);
        if (r0 > 0.f && r0 < 1.f) { tq[n] = r0; n++; }
        if (r1 > 0.f && r1 < 1.f && r1 != r0) { tq[n] = r1; n++; }
    } else if (c.type == CT_RATIONAL) {
        const float w0 = 1.f, w1 = c.w, w2 = 1.f;
        float p0 = w0 * v0, p1 = w1 * v1, p2 = w2 * v2;
        float pw01 = p0 * w1 - p1 * w0;
        float pw12 = p1 * w2 - p2 * w1;
        float pw20 = p2 * w0 - p0 * w2;
        float r0 = 0.f, r1 = 0.f;
        solve_quad(pw01 + pw12 + pw20, -(2.f * pw01 + pw20), pw01, r0, r1);
        if (r0 > 0.f && r0 < 1.f) { tq[n] = r0; n++; }
        if (r1 > 0.f && r1 < 1.f && r1 != r0) { tq[n] = r1; n++; }
    }
}

// d_get_xy_begin_end_delta + d_udpate_cut_range (ras_cut.h:693-777)
struct CutRange {
    int32_t xb, xe, yb, ye, nx, ny;
    float dx, dy;
};
__device__ __forceinline__ CutRange cut_range(float v0x, float v0y, float v1x, float v1y, int W, int H) {
    CutRange r;
    if (v0x <= v1x) { r.xb = wadd(floor_even(v0x), 2); r.xe = floor_even(v1x); r.dx = 2.f; }
    else { r.xb = wadd(floor_even(v1x), 2); r.xe = floor_even(v0x); r.dx = -2.f; }
    if (v0y <= v1y) { r.yb = wadd(floor_even(v0y), 2); r.ye = floor_even(v1y); r.dy = 2.f; }
    else { r.yb = wadd(floor_even(v1y), 2); r.ye = floor_even(v0y); r.dy = -2.f; }
    const int32_t xmax = (W & ~1) + 2, ymax = (H & ~1) + 2;
    if ((r.xb < 0 && r.xe < 0) || (r.xb > xmax && r.xe > xmax) || (r.xb > r.xe)) {
        r.nx = 0;
    } else {
        r.xb = tmin(tmax(r.xb, 0), xmax);
        r.xe = tmin(tmax(r.xe, 0), xmax);
        r.nx = tmax((r.xe - r.xb) / 2 + 1, 0);
    }
    if ((r.yb < 0 && r.ye < 0) || (r.yb > ymax && r.ye > ymax) || (r.yb > r.ye)) {
        r.ny = 0;
    } else {
        r.yb = tmin(tmax(r.yb, 0), ymax);
        r.ye = tmin(tmax(r.ye, 0), ymax);
        r.ny = tmax((r.ye - r.yb) / 2 + 1, 0);
    }
    return r;
}

__device__ __forceinline__ float pick5(int i, float a, float b, float c, float d, float e) {
    return i == 0 ? a : (i == 1 ? b : (i == 2 ? c : (i == 3 ? d : e)));
}

// k_make_intersection_0 (ras_cut.h:1254-1482): monotone cuts, then per monotone piece the
// numbers of even x / y cut lines it crosses (d_udpate_cut_range) and the curve's fragment
// count.  Also the number of solve chains (two per piece) of the intersection pass.
__device__ __forceinline__ int wave_min_i(int v) { return wave_reduce(v, INT_MAX, OpMin()); }
__device__ __forceinline__ int wave_max_i(int v) { return wave_reduce(v, INT_MIN, OpMax()); }

// Range of cell rows a visible curve's fragments can fall in: a fragment's row comes from
// its chord midpoint, which lies inside the control-point hull (rationals with w > 0), so
// the hull's rows with one row of margin for rounding, clamped to the canvas rows.
__device__ __forceinline__ void curve_rows(const Curve &cu, int H, int &rlo, int &rhi) {
    const int nv = cu.type & 7;
    float lo = fminf(cu.y0, cu.y1), hi = fmaxf(cu.y0, cu.y1);
    if (nv > 2) { lo = fminf(lo, cu.y2); hi = fmaxf(hi, cu.y2); }
    if (nv > 3) { lo = fminf(lo, cu.y3); hi = fmaxf(hi, cu.y3); }
    const int rmax = (H - 1) >> 1;
    const bool hull = cu.type != CT_RATIONAL || cu.w > 0.f;
    if (hull && fabsf(lo) < 1e30f && fabsf(hi) < 1e30f) {
        rlo = tmax((floor_i32(lo) >> 1) - 1, 0);
        rhi = tmin((floor_i32(hi) >> 1) + 1, rmax);
    } else {
        rlo = 0;
        rhi = rmax;
    }
}

__global__ void __launch_bounds__(256) k_monotone(SceneDev sc, const float2 *__restrict__ tv, const uint32_t *__restrict__ pflags,
                                                   int W, int H, float4 *crec, uint32_t *cfrag,
                                                   uint32_t *pcnt, uint32_t *nchain, int2 *prow) {
    // the block's 64-byte curve records, staged so that they are stored with consecutive lanes
    __shared__ float4 stg[256 * 4];
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = c < sc.C;
    bool vis = false;
    int rlo = 0, rhi = -1;
    uint32_t path = 0u;
    if (live) {
        Curve cu = load_curve(sc, tv, c);
        path = sc.cinfo[c].y;
        vis = region_visible(pflags[path]);
        path_canvas(sc, path, W, H);
        float tq[4] = {0.f, 0.f, 0.f, 0.f};
        int n = 0;
        if (vis) {
            monotone_axis(cu, cu.x0, cu.x1, cu.x2, cu.x3, tq, n);
            monotone_axis(cu, cu.y0, cu.y1, cu.y2, cu.y3, tq, n);
        }
        float q0 = tq[0], q1 = tq[1], q2 = tq[2], q3 = tq[3];
        if (n >= 2) { if (q1 < q0) { float t = q0; q0 = q1; q1 = t; } }
        if (n >= 3) {
            float t2 = q2, t1 = q1;
            if (t2 < t1) {
                q2 = t1;
                float t0 = q0;
                if (t2 < t0) { q1 = t0; q0 = t2; } else { q1 = t2; }
            }
        }
        if (n >= 4) {
            float t3 = q3, t2 = q2;
            if (t3 < t2) {
                q3 = t2;
                float t1 = q1;
                if (t3 < t1) {
                    q2 = t1;
                    float t0 = q0;
                    if (t3 < t0) { q1 = t0; q0 = t3; } else { q1 = t3; }
                } else {
                    q2 = t3;
                }
            }
        }
        stg[4 * threadIdx.x] = make_float4(cu.x0, cu.y0, cu.x1, cu.y1);
        stg[4 * threadIdx.x + 1] = make_float4(cu.x2, cu.y2, cu.x3, cu.y3);
        stg[4 * threadIdx.x + 2] = make_float4(q0, q1, q2, q3);
        stg[4 * threadIdx.x + 3] = make_float4(bf((uint32_t)cu.type | ((uint32_t)n << 8)), cu.w, bf(path),
                                               bf(sc.cinfo[c].z >> 8));
        uint32_t cnt = 0;
        uint32_t pc[5] = {0u, 0u, 0u, 0u, 0u};
        const int npieces = vis ? n + 1 : 0;
        if (vis) {
            float v0x = cu.x0, v0y = cu.y0;
            for (int ms = 0; ms < npieces; ++ms) {
                float t1 = (ms == n) ? 1.f : pick5(ms, q0, q1, q2, q3, 1.f);
                float v1x = ex(cu, t1), v1y = ey(cu, t1);
                CutRange r = cut_range(v0x, v0y, v1x, v1y, W, H);
                cnt += 1u + (uint32_t)r.nx + (uint32_t)r.ny;
                pc[ms] = (uint32_t)r.nx | ((uint32_t)r.ny << 16);
                v0x = v1x; v0y = v1y;
            }
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) pcnt[5 * (size_t)c + k] = pc[k];
        cfrag[c] = cnt;
        nchain[c] = 2u * (uint32_t)npieces;
        if (vis) curve_rows(cu, H, rlo, rhi);
    }
    __syncthreads();
    const uint32_t c0 = blockIdx.x * blockDim.x;
    const uint32_t nrec = 4u * (sc.C - c0 < blockDim.x ? sc.C - c0 : blockDim.x);
    for (uint32_t k = threadIdx.x; k < nrec; k += blockDim.x) crec[4 * (size_t)c0 + k] = stg[k];
    // the path's row range, one atomic pair per distinct path of the wave
    const int lane = threadIdx.x & 63;
    uint64_t pend = __ballot(vis && rlo <= rhi);
    while (pend) {
        const int leader = __ffsll((long long)pend) - 1;
        const uint32_t lp = (uint32_t)__builtin_amdgcn_readlane((int)path, leader);
        const bool mine = ((pend >> lane) & 1ull) && path == lp;
        const uint64_t grp = __ballot(mine);
        const int mn = wave_min_i(mine ? rlo : INT_MAX), mx = wave_max_i(mine ? rhi : INT_MIN);
        if (lane == leader) {
            atomicMin(&prow[lp].x, mn);
            atomicMax(&prow[lp].y, mx);
        }
        pend &= ~grp;
    }
}

// Work lists.  Pieces (curve << 3 | piece) with nx + ny + 1 >= 128 cuts (cubic ones from
// cubic_min cuts, see launch_intersect) are "long": their two solve chains (curve << 4 |
// piece << 1 | side, non-empty only) are listed, and the piece for the wave-parallel merge.  Shorter pieces are listed for
// one thread that solves and walks both sides.  Chains and short pieces are grouped by
// (cubic or closed-form solve, length bin), longest first, so the lanes of a wave run
// loops of the same kind and about the same trip count and the long sequential walks
// start early.  Blocks of a fixed number take runs of curves: a count pass leaves each block's
// entries per class, and in the place pass every block sums the counts before its own (its
// first place in each class) and hands out places with LDS atomics.  (With one device atomic
// per class and block of 1024 curves instead, the two passes waited for the same hundred
// addresses: 84 and 92 us on a sheet of 100000 glyph paths, now 40 and 61.)
constexpr int kLenBins = 25;
constexpr int kChainClasses = 2 * kLenBins;                     // cubic bins, then closed-form bins
constexpr int kLongPieceClass = kChainClasses;                  // one class
constexpr int kShortClass0 = kChainClasses + 1;                 // cubic bins, then closed-form bins
constexpr int kListClasses = kShortClass0 + 2 * kLenBins;
constexpr uint32_t kLongPiece = 128;
constexpr int kChainListThreads = 1024;
constexpr uint32_t kListBlocks = 512;
// Frame::lcount: class counts, then their exclusive sums over all classes and the total, then
// how many chains at the list's front are solved by several lanes each
constexpr int kListPre = kListClasses;
constexpr int kListWide = kListPre + kListClasses + 1;
static_assert((kListWide + 1) * sizeof(uint32_t) <= kListCountBytes, "class counts exceed their buffer");

// Length bins, longest first.  Below 256 a bin's longest entry is at most 4/3 of its
// shortest, so that the lanes of a wave run loops of nearly equal trip counts.  The bin
// of L is the number of lower bounds above L.
#define SL_BIN_LOWER {384, 256, 192, 160, 128, 112, 96, 80, 65, 57, 49, 41, 33, 29, 25, 21, 17, 13, 9, 7, 5, 4, 3, 2, 1}
__device__ __forceinline__ int len_bin(uint32_t L) {
    constexpr uint32_t lower[kLenBins] = SL_BIN_LOWER;
    int b = 0;
#pragma unroll
    for (int i = 0; i < kLenBins; ++i) b += lower[i] > L ? 1 : 0;
    return b;
}
// the shortest length of bin b, 0 beyond the last
__device__ __forceinline__ uint32_t bin_lower(int b) {
    constexpr uint32_t lower[kLenBins] = SL_BIN_LOWER;
    uint32_t v = 0u;
#pragma unroll
    for (int i = 0; i < kLenBins; ++i) v = b == i ? lower[i] : v;
    return v;
}
#undef SL_BIN_LOWER

struct CurvePieces {
    int np;
    int cb;  // 0 for a cubic, kLenBins otherwise
    uint32_t pc[5];
};

__device__ __forceinline__ CurvePieces curve_pieces(const SceneDev &sc, uint32_t C, uint32_t c,
                                                    const uint32_t *__restrict__ nchain,
                                                    const uint32_t *__restrict__ pcnt) {
    CurvePieces r;
    const bool live = c < C;
    r.np = live ? (int)(nchain[c] >> 1) : 0;
    r.cb = (live && sc.ctype[c] == CT_CUBIC) ? 0 : kLenBins;
#pragma unroll
    for (int k = 0; k < 5; ++k) r.pc[k] = k < r.np ? pcnt[5 * (size_t)c + k] : 0u;
    return r;
}

// the classes of piece k's entries: x chain, y chain (-1 when not listed), piece
__device__ __forceinline__ void piece_classes(const CurvePieces &cp, int k, uint32_t cubic_min, int &qx, int &qy,
                                              int &qp) {
    const uint32_t nx = cp.pc[k] & 0xFFFFu, ny = cp.pc[k] >> 16, L = nx + ny + 1;
    if (L >= (cp.cb ? kLongPiece : cubic_min)) {
        qx = nx ? cp.cb + len_bin(nx) : -1;
        qy = ny ? cp.cb + len_bin(ny) : -1;
        qp = kLongPieceClass;
    } else {
        qx = qy = -1;
        qp = kShortClass0 + cp.cb + len_bin(L);
    }
}

// adds the classes of curves [c0, c1) to h
__device__ __forceinline__ void count_classes(const SceneDev &sc, uint32_t C, uint32_t c0, uint32_t c1,
                                              const uint32_t *__restrict__ nchain, const uint32_t *__restrict__ pcnt,
                                              uint32_t cubic_min, uint32_t *h) {
    for (uint32_t c = c0 + threadIdx.x; c < c1; c += kChainListThreads) {
        const CurvePieces cp = curve_pieces(sc, C, c, nchain, pcnt);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            if (k >= cp.np) break;
            int qx, qy, qp;
            piece_classes(cp, k, cubic_min, qx, qy, qp);
            if (qx >= 0) atomicAdd(&h[qx], 1u);
            if (qy >= 0) atomicAdd(&h[qy], 1u);
            atomicAdd(&h[qp], 1u);
        }
    }
}

// blk[class * blocks + block]: the block's entries of the class; a block takes `per` curves
__global__ void __launch_bounds__(kChainListThreads) k_list_count(SceneDev sc, uint32_t C, uint32_t per,
                                                                  const uint32_t *__restrict__ nchain,
                                                                  const uint32_t *__restrict__ pcnt, uint32_t cubic_min,
                                                                  uint32_t *__restrict__ blk) {
    __shared__ uint32_t h[kListClasses];
    for (int q = threadIdx.x; q < kListClasses; q += blockDim.x) h[q] = 0u;
    __syncthreads();
    const uint32_t c0 = blockIdx.x * per, c1 = c0 + per < C ? c0 + per : C;
    count_classes(sc, C, c0, c1, nchain, pcnt, cubic_min, h);
    __syncthreads();
    for (int q = threadIdx.x; q < kListClasses; q += blockDim.x) blk[(size_t)q * gridDim.x + blockIdx.x] = h[q];
}

// Which cubic chains get several lanes each: those of the first `bins` length bins, as long as
// their cuts (by the bins' shortest lengths) are no more than `load` chains of the longest bin
// there is would have (launch_intersect has the limits).
struct WideRule {
    int bins;
    uint32_t load;
};

// Lists from the block counts (at most kListBlocks); writes the class counts and their sums.
// SOLO: one block, which counts for itself first.
template <bool SOLO>
__global__ void __launch_bounds__(kChainListThreads) k_list_place(SceneDev sc, uint32_t C, uint32_t per,
                                                                  const uint32_t *__restrict__ nchain,
                                                                  const uint32_t *__restrict__ pcnt,
                                                                  const uint32_t *__restrict__ coff, uint32_t cubic_min,
                                                                  WideRule rule, const uint32_t *__restrict__ blk,
                                                                  uint32_t *__restrict__ cnt, uint4 *clist, uint4 *plist) {
    __shared__ uint32_t total[kListClasses], base[kListClasses];
    constexpr int kWaves = kChainListThreads / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (SOLO) {
        for (int q = threadIdx.x; q < kListClasses; q += kChainListThreads) total[q] = base[q] = 0u;
        __syncthreads();
        count_classes(sc, C, 0u, C, nchain, pcnt, cubic_min, total);
    } else {
        const uint32_t nb = gridDim.x;
#pragma unroll
        for (int j = 0; j < (kListClasses + kWaves - 1) / kWaves; ++j) {
            const int q = j * kWaves + w;
            if (q >= kListClasses) break;
            uint32_t tot = 0u, before = 0u;
#pragma unroll
            for (uint32_t i0 = 0; i0 < kListBlocks; i0 += 64) {
                const uint32_t i = i0 + (uint32_t)lane;
                const uint32_t v = i < nb ? blk[(size_t)q * nb + i] : 0u;
                tot += v;
                before += i < blockIdx.x ? v : 0u;
            }
            tot = (uint32_t)wave_reduce((int)tot, 0, OpAdd());
            before = (uint32_t)wave_reduce((int)before, 0, OpAdd());
            if (lane == 0) { total[q] = tot; base[q] = before; }
        }
    }
    __syncthreads();
    // class offsets: within the chain list, and within the piece list (long pieces first)
    if (w < 2) {
        const int q = w * kChainClasses + lane, n = w ? kListClasses - kChainClasses : kChainClasses;
        const uint32_t v = lane < n ? total[q] : 0u, inc = wave_incl_scan(v);
        if (lane < n) {
            base[q] += inc - v;
            if (blockIdx.x == 0) {
                cnt[q] = v;
                cnt[kListPre + q] = inc - v;
                if (q == kListClasses - 1) cnt[kListPre + kListClasses] = inc;
            }
        }
    }
    __syncthreads();
    if (w == kWaves - 1 && blockIdx.x == gridDim.x - 1) {  // the wave with the fewest curves
        const uint32_t v = lane < kLenBins ? total[lane] : 0u, len = bin_lower(lane);
        const uint64_t some = __ballot(v != 0u), cuts = (uint64_t)v * len;
        const uint32_t longest = some ? (uint32_t)__builtin_amdgcn_readlane((int)len, (int)__builtin_ctzll(some)) : 0u;
        const uint32_t chains = wave_incl_scan(v);
        const uint32_t sum = wave_incl_scan(cuts < (1u << 26) ? (uint32_t)cuts : 1u << 26);  // 25 of them fit
        const int b = (int)__builtin_ctzll(~__ballot(lane < rule.bins && sum <= rule.load * longest));
        const uint32_t wide = b ? (uint32_t)__builtin_amdgcn_readlane((int)chains, b - 1) : 0u;
        if (lane == 0) cnt[kListWide] = wide;
    }
    const uint32_t c0 = blockIdx.x * per, c1 = c0 + per < C ? c0 + per : C;
    for (uint32_t c = c0 + threadIdx.x; c < c1; c += kChainListThreads) {
        const CurvePieces cp = curve_pieces(sc, C, c, nchain, pcnt);
        uint32_t off = cp.np ? coff[c] : 0u;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            if (k >= cp.np) break;
            int qx, qy, qp;
            piece_classes(cp, k, cubic_min, qx, qy, qp);
            // each entry carries its piece's ts offset and cut counts, so that the intersection
            // passes read only the curve's record besides it
            const uint32_t pb = off, pw = cp.pc[k];
            off += 1u + (pw & 0xFFFFu) + (pw >> 16);
            if (qx >= 0) clist[atomicAdd(&base[qx], 1u)] = make_uint4((c << 4) | ((uint32_t)k << 1), pb, pw, 0u);
            if (qy >= 0) clist[atomicAdd(&base[qy], 1u)] = make_uint4((c << 4) | ((uint32_t)k << 1) | 1u, pb, pw, 0u);
            plist[atomicAdd(&base[qp], 1u)] = make_uint4((c << 3) | (uint32_t)k, pb, pw, 0u);
        }
    }
}

__device__ __forceinline__ uint32_t chain_total(const uint32_t *__restrict__ cnt) {
    return cnt[kListPre + kChainClasses - 1] + cnt[kChainClasses - 1];
}

// t | flags of a monotone piece's end: low bits 2 when the end lies on an integral x,
// else 3 (k_make_intersection_impl_1, ras_cut.h:858-865)
__device__ __forceinline__ float piece_end_flags(float t_raw, float vx) {
    float t = bf(fb(t_raw) & 0xFFFFFFFCu);
    if (floorf(vx) == vx) return bf((fb(t) & 0xFFFFFFFCu) | 2u);
    return bf(fb(t) | 3u);
}

// One cut solve on one coordinate of the curve (ras_cut.h:1004-1106): line and
// quadratic / rational in closed form, cubic by 24-step bisection from t_min.
__device__ __forceinline__ float solve_cut(int type, float w, float a0, float a1, float a2, float a3, float cc,
                                           float t_min, float t1) {
    if (type == CT_LINEAR) return tmin(tmax((cc - a0) * safe_rcp(a1 - a0), t_min), t1);
    if (type == CT_QUAD) return solve_quad_bezier(a0, a1, a2, cc, t_min, t1);
    if (type == CT_RATIONAL) return solve_quad_bezier(a0 - cc, (a1 - cc) * w, a2 - cc, 0.f, t_min, t1);
    // 24 bisection steps.  An end moves only to a midpoint whose f - cc has the sign bit of its
    // own (f - cc is negative exactly when f < cc), so the ends are kept by their side of cc:
    // the midpoint of the two is the same whichever is the lower one.
    const float vlo = curve_eval(CT_CUBIC, 0.f, a0, a1, a2, a3, t_min);
    float t_solve = t_min;
    if (vlo != cc) {
        float p = vlo < cc ? t_min : t1, q = vlo < cc ? t1 : t_min;
        float last_v = 0.f;
        for (int it = 0; it < 24; ++it) {
            const float tm = (p + q) * .5f;
            const float vm = curve_eval(CT_CUBIC, 0.f, a0, a1, a2, a3, tm);
            const bool low = vm < cc;
            p = low ? tm : p;
            q = low ? q : tm;
            t_solve = tm;
            last_v = vm;
        }
        if (fabsf(last_v - cc) > 1.f) t_solve = t_min;
    }
    return t_solve;
}

// The cut solve state of one side of a monotone piece.  In the reference's merge walk
// (ras_cut.h:910-1232) the j-th cut on one side is solved from the t the same side
// produced last (or the piece start), so each side's chain is independent of the other
// side's and is solved in order, each t stored as t | side.
struct SideSolver {
    float a0, a1, a2, a3, cc, dd, t_min, t1m, w;
    int type;
    uint32_t side;
    __device__ __forceinline__ float next() {
        const float t = solve_cut(type, w, a0, a1, a2, a3, cc, t_min, t1m);
        const float tm = bf((fb(t) & 0xFFFFFFFCu) | side);
        t_min = tm;
        cc += dd;
        return tm;
    }
};

struct PieceSetup {
    uint32_t c, base, nx, ny;
    float t0m;
    SideSolver sx, sy;
};

// piece k of curve c: its ts offset, cut counts, start flags and both sides' solvers
// (e: the work-list entry {curve and piece, ts offset of the piece, nx | ny << 16})
__device__ __forceinline__ PieceSetup piece_setup(const SceneDev &sc, const float4 *__restrict__ crec,
                                                  uint32_t c, int k, uint4 e, int W, int H) {
    PieceSetup p;
    p.c = c;
    p.base = e.y;
    p.nx = e.z & 0xFFFFu;
    p.ny = e.z >> 16;
    const CurveRec rec = load_rec(crec, c);
    path_canvas(sc, rec.path, W, H);
    const Curve &cu = rec.cu;
    const float4 q = rec.q;
    const int n = rec.n;
    float v0x = cu.x0, v0y = cu.y0, t0m = 0.f;
    if (k > 0) {
        const float tr = pick5(k - 1, q.x, q.y, q.z, q.w, 1.f);
        v0x = ex(cu, tr);
        v0y = ey(cu, tr);
        t0m = piece_end_flags(tr, v0x);
    }
    p.t0m = t0m;
    const float t1r = (k == n) ? 1.f : pick5(k, q.x, q.y, q.z, q.w, 1.f);
    const float v1x = ex(cu, t1r), v1y = ey(cu, t1r);
    const float t1m = piece_end_flags(t1r, v1x);
    const CutRange r = cut_range(v0x, v0y, v1x, v1y, W, H);
    p.sx.a0 = cu.x0; p.sx.a1 = cu.x1; p.sx.a2 = cu.x2; p.sx.a3 = cu.x3;
    p.sx.cc = (float)(r.dx < 0.f ? r.xe : r.xb);
    p.sx.dd = r.dx;
    p.sy.a0 = cu.y0; p.sy.a1 = cu.y1; p.sy.a2 = cu.y2; p.sy.a3 = cu.y3;
    p.sy.cc = (float)(r.dy < 0.f ? r.ye : r.yb);
    p.sy.dd = r.dy;
    p.sx.t_min = p.sy.t_min = t0m;
    p.sx.t1m = p.sy.t1m = t1m;
    p.sx.w = p.sy.w = cu.w;
    p.sx.type = p.sy.type = cu.type;
    p.sx.side = 0u;
    p.sy.side = 1u;
    return p;
}

// Intersection pass 1, long pieces: one thread per (curve, piece, side) chain, the t's
// stored for the merge pass (k_merge_long) with 16-byte stores.
__device__ __forceinline__ void solve_chain(const SceneDev &sc, const float4 *__restrict__ crec, uint4 e, int W,
                                            int H, float *chain_t) {
    const uint32_t d = e.x;
    const int side = (int)(d & 1u);
    PieceSetup p = piece_setup(sc, crec, d >> 4, (int)((d >> 1) & 7u), e, W, H);
    const uint32_t cnt = side ? p.ny : p.nx;
    SideSolver sv = side ? p.sy : p.sx;
    float *out = chain_t + p.base + (side ? p.nx : 0u);
    // scalar stores up to a 16-byte boundary, then whole float4 stores, then the tail
    const uint32_t head = (uint32_t)((4u - (((uintptr_t)out >> 2) & 3u)) & 3u);
    float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t j = 0; j < cnt; ++j) {
        const float tm = sv.next();
        if (j < head) {
            out[j] = tm;
        } else {
            const uint32_t ph = (j - head) & 3u;
            if (ph == 0) q4.x = tm;
            else if (ph == 1) q4.y = tm;
            else if (ph == 2) q4.z = tm;
            else q4.w = tm;
            if (ph == 3) *(float4 *)(out + j - 3) = q4;
        }
    }
    if (cnt > head) {
        const uint32_t rem = (cnt - head) & 3u;  // values still held in q4
        const uint32_t j0 = cnt - rem;
        if (rem > 0) out[j0] = q4.x;
        if (rem > 1) out[j0 + 1] = q4.y;
        if (rem > 2) out[j0 + 2] = q4.z;
    }
}

// Cubic chains of frames that leave the GPU idle.  A chain is serial: every cut's bisection
// starts from the previous cut's t, and its 24 steps depend on each other, so one lane needs
// about 1.5 us a cut and a frame's longest chain sets the pass's time whatever the size of
// the GPU.  Here 2^K lanes share a chain: lane l follows the bits of l through K halvings,
// computing the interval ends exactly as the serial steps would, evaluates the curve at its
// lower end T[l] (T[1] .. T[2^K - 1] are the 2^K - 1 midpoints the next K steps can visit), and
// the steps' outcome is read from all lanes' signs at once.  Along a monotone piece the signs
// change once, and the interval left is the one between the last T on the lower side and the
// first on the upper; where rounding makes them change more often, the K steps are walked
// through the sign bits one by one.  Either way the result is the serial bisection's, bit for bit.
struct WideChain {
    float a0, a1, a2, a3, d01, d12, d23;
    __device__ __forceinline__ float eval(float t) const {  // curve_eval of a cubic, its first differences at hand
        const float q0 = a0 + t * d01, q1 = a1 + t * d12, q2 = a2 + t * d23;
        const float l0 = q0 + t * (q1 - q0), l1 = q1 + t * (q2 - q1);
        return l0 + t * (l1 - l0);
    }
};

template <int CTRL> __device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xf, 0xf, false);
}
// row-wide (16 lanes) maximum / minimum in every lane of the row
__device__ __forceinline__ uint32_t row_max(uint32_t x) {
    x = tmax(x, dpp_u32<0x128>(x));  // row_ror:8, 4, 2, 1
    x = tmax(x, dpp_u32<0x124>(x));
    x = tmax(x, dpp_u32<0x122>(x));
    return tmax(x, dpp_u32<0x121>(x));
}
__device__ __forceinline__ uint32_t row_min(uint32_t x) {
    x = tmin(x, dpp_u32<0x128>(x));
    x = tmin(x, dpp_u32<0x124>(x));
    x = tmin(x, dpp_u32<0x122>(x));
    return tmin(x, dpp_u32<0x121>(x));
}

// T[l] of the next K steps from the interval [lo, hi], 0 <= lo <= hi.  The interval is kept
// scaled by 2^k at step k, so a midpoint is a plain sum S = A + B (its rounding does not depend
// on the scale) and the next one S + 2 X, X being the end the step keeps: one fma a step on the
// critical path.
template <int K> __device__ __forceinline__ float wide_node(float lo, float hi, int l) {
    float S = lo + hi, A = lo, X = (l >> (K - 1)) & 1 ? hi : lo;
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
        const bool up = (l >> k) & 1;
        const float A2 = A + A;
        if (k > 0) {
            const bool same = ((l >> k) & 1) == ((l >> (k - 1)) & 1);
            const float S2 = __builtin_fmaf(X, 2.f, S), X2 = X + X;
            X = same ? X2 : S;
            A = up ? S : A2;
            S = S2;
        } else {
            A = up ? S : A2;
        }
    }
    return A * (1.f / (float)(1 << K));
}

// One cut by a whole wave, four rounds of six steps; `odd` is set where the signs changed more
// than once (the result is then not to be used).
__device__ __forceinline__ float wide_cut64(const WideChain &w, float cc, float t_min, float t1, bool &odd) {
    const int lane = threadIdx.x & 63;
    float lo = t_min, hi = t1;
    uint64_t flip = 0ull, spread = 0ull, eq = 0ull, far = 0ull;
    uint32_t leaf = 0u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float T = wide_node<6>(lo, hi, lane);
        const float Th = lane == 0 ? hi : T;  // the upper end of leaf 63 is the interval's
        const float v = w.eval(T);
        uint64_t m = __ballot(v < cc);
        if (r == 0) {
            eq = __ballot(v == cc) & 1ull;       // lane 0 is at t_min
            flip = (m & 1ull) ? 0ull : ~0ull;    // lanes on t_min's side get a 1
        }
        m = (m ^ flip) | 1ull;
        spread |= m & (m + 1ull);
        leaf = (uint32_t)__popcll(m) - 1u;
        if (r == 3) far = __ballot(fabsf(v - cc) > 1.f);
        lo = bf((uint32_t)__builtin_amdgcn_readlane((int)fb(T), leaf));
        hi = bf((uint32_t)__builtin_amdgcn_readlane((int)fb(Th), (leaf + 1u) & 63u));
    }
    odd = spread != 0ull;
    const float t = (leaf & 1u) ? lo : hi;  // the last midpoint
    return (eq || ((far >> (leaf | 1u)) & 1ull)) ? t_min : t;
}

// One cut by each of the wave's four rows of 16 lanes: six rounds of four steps.
__device__ __forceinline__ float wide_cut16(const WideChain &w, float cc, float t_min, float t1, bool &odd) {
    const int lane = threadIdx.x & 63, sub = lane & 15;
    float lo = t_min, hi = t1;
    bool below = false, exact = false;
    uint32_t rows = 0u, far = 0u;
    odd = false;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        const float T = wide_node<4>(lo, hi, sub);
        const float v = w.eval(T);
        if (r == 0) {
            const float v0 = bf(dpp_u32<0x150>(fb(v)));  // row_newbcast:0, at t_min
            exact = v0 == cc;
            below = v0 < cc;
        }
        const bool up = (v < cc) == below || sub == 0;
        // t >= 0: the bits order like the values
        const uint32_t cl = row_max(up ? fb(T) : fb(lo)), ch = row_min(up ? fb(hi) : fb(T));
        odd |= cl > ch;
        if (r == 5) {
            // the row's sign bits give the last midpoint: the lower end left after an up step
            const uint64_t mu = __ballot(up), mf = __ballot(fabsf(v - cc) > 1.f);
            const int sh = lane & 16;
            rows = (((lane & 32) ? (uint32_t)(mu >> 32) : (uint32_t)mu) >> sh) & 0xFFFFu;
            far = (((lane & 32) ? (uint32_t)(mf >> 32) : (uint32_t)mf) >> sh) & 0xFFFFu;
        }
        lo = bf(cl);
        hi = bf(ch);
    }
    const uint32_t leaf = (uint32_t)__popc(rows) - 1u;
    return (exact || ((far >> (leaf | 1u)) & 1u)) ? t_min : ((leaf & 1u) ? lo : hi);
}

// Chains [0, n) of the list (cubic, longest first) over the waves of `blocks` blocks: the
// first n64 of them a wave each, the others four to a wave, the long ones at a raised wave
// priority, since the last of them ends the pass.  The t's of a chain are stored a row or a
// wave at a time.  Bound by the instructions of a chain's own wave (about 250 a cut with 64
// lanes, 300 with 16, against 528 with one lane).  Rows of 16 lanes with four nodes a lane
// (four rounds of six steps) were slower: 1.27 us a cut for 1.06.
__device__ __forceinline__ void wide_chains(const SceneDev &sc, const float4 *__restrict__ crec,
                                            const uint4 *__restrict__ clist, uint32_t n, uint32_t blocks,
                                            int W, int H, float *__restrict__ chain_t) {
    const int lane = threadIdx.x & 63;
    const uint32_t waves = blocks * (blockDim.x >> 6);
    const uint32_t wave = (threadIdx.x >> 6) * blocks + blockIdx.x;  // neighbours in the list go to other CUs
    // with few chains, the longest of them a wave each: 0.67 us a cut against 1.06 us
    const uint32_t n64 = n <= 8192u ? tmin(512u, n) : 0u;
    const uint32_t units = n64 + (n - n64 + 3u) / 4u;
    for (uint32_t u = wave; u < units; u += waves) {
        const bool whole = u < n64;
        const uint32_t i = whole ? u : n64 + 4u * (u - n64) + (uint32_t)(lane >> 4);
        const bool live = i < n;
        const uint4 e = clist[live ? i : 0u];
        const int side = (int)(e.x & 1u);
        const PieceSetup p = piece_setup(sc, crec, e.x >> 4, (int)((e.x >> 1) & 7u), e, W, H);
        const SideSolver sv = side ? p.sy : p.sx;
        const uint32_t cnt = live ? (side ? p.ny : p.nx) : 0u;
        float *out = chain_t + p.base + (side ? p.nx : 0u);
        const WideChain w{sv.a0, sv.a1, sv.a2, sv.a3, sv.a1 - sv.a0, sv.a2 - sv.a1, sv.a3 - sv.a2};
        const bool tiny = !(sv.t1m >= 1e-30f);  // scaled sums would round subnormals differently
        float cc = sv.cc, t = sv.t_min, keep = 0.f;
        if (whole) {
            __builtin_amdgcn_s_setprio(3);
            for (uint32_t j = 0; j < cnt; ++j) {
                bool odd;
                float r = wide_cut64(w, cc, t, sv.t1m, odd);
                if (odd || tiny) r = solve_cut(CT_CUBIC, 0.f, sv.a0, sv.a1, sv.a2, sv.a3, cc, t, sv.t1m);
                t = bf((fb(r) & 0xFFFFFFFCu) | sv.side);
                cc += sv.dd;
                keep = (j & 63u) == (uint32_t)lane ? t : keep;
                if ((j & 63u) == 63u || j + 1 == cnt) {
                    const uint32_t j0 = j & ~63u;
                    if (j0 + lane <= j) out[j0 + lane] = keep;
                }
            }
        } else {
            const uint32_t most = (uint32_t)wave_reduce((int)cnt, 0, OpMaxU());
            const uint32_t sub = (uint32_t)(lane & 15);
            if (most > 64u) __builtin_amdgcn_s_setprio(2);
            else __builtin_amdgcn_s_setprio(1);
            for (uint32_t j = 0; j < most; ++j) {
                bool odd;
                float r = wide_cut16(w, cc, t, sv.t1m, odd);
                if (__ballot(odd || tiny)) {
                    const float q = solve_cut(CT_CUBIC, 0.f, sv.a0, sv.a1, sv.a2, sv.a3, cc, t, sv.t1m);
                    r = odd || tiny ? q : r;
                }
                t = bf((fb(r) & 0xFFFFFFFCu) | sv.side);
                cc += sv.dd;
                keep = (j & 15u) == sub ? t : keep;
                const uint32_t k = (j & ~15u) + sub;
                if (((j & 15u) == 15u || j + 1 == most) && k <= j && k < cnt) out[k] = keep;
            }
        }
        __builtin_amdgcn_s_setprio(0);
    }
}

// Intersection pass 2 replays the reference's slot walk (ras_cut.h:910-1000) per
// monotone piece over the piece's solved chains: pick the x slot when x <= y, emit its t,
// refill it from the chain or with the exhausted marker 2 | side; equal consecutive t's
// OR their flags into the previous entry.  A piece starts at the previous piece's end
// flags (t = 0 for the first), exactly as the per-curve walk carries them.
struct PieceRef {
    uint32_t c, base, nx, ny;
    float t0m;
};

__device__ __forceinline__ PieceRef piece_ref(const float4 *__restrict__ crec, uint4 e) {
    PieceRef r;
    const uint32_t d = e.x;
    r.c = d >> 3;
    const int k = (int)(d & 7u);
    r.base = e.y;
    r.nx = e.z & 0xFFFFu;
    r.ny = e.z >> 16;
    r.t0m = 0.f;
    if (k > 0) {
        const CurveRec rec = load_rec(crec, r.c);
        const float tr = pick5(k - 1, rec.q.x, rec.q.y, rec.q.z, rec.q.w, 1.f);
        r.t0m = piece_end_flags(tr, ex(rec.cu, tr));
    }
    return r;
}

// Sequential reader of a chain: one 16-byte load per aligned group of four values (the
// chain buffer is 16-byte aligned and padded, so whole groups stay inside it).
struct ChainReader {
    const float *p;
    const float4 *blk;
    float4 buf;
    __device__ __forceinline__ void init(const float *q) {
        p = q;
        blk = nullptr;
    }
    __device__ __forceinline__ float at(uint32_t i) {
        const uintptr_t a = (uintptr_t)(p + i);
        const float4 *b = (const float4 *)(a & ~(uintptr_t)15);
        if (b != blk) {
            blk = b;
            buf = *b;
        }
        const uint32_t c = (uint32_t)(a >> 2) & 3u;
        return c == 0 ? buf.x : (c == 1 ? buf.y : (c == 2 ? buf.z : buf.w));
    }
};

__device__ __forceinline__ void walk_piece(const PieceRef &r, const float *__restrict__ chain_t, int2 *ts) {
    int2 *out = ts + r.base;
    const uint32_t nx = r.nx, ny = r.ny;
    ChainReader X, Y;
    X.init(chain_t + r.base);
    Y.init(chain_t + r.base + nx);
    const float t0m = r.t0m;
    const float two = 2.f, two1 = bf(fb(2.f) | 1u);
    float xs, ys;
    uint32_t xi = 0, yi = 0, rx, ry;
    if (nx == 0) { xs = two; ys = t0m; rx = 0; ry = ny; }
    else if (ny == 0) { xs = t0m; ys = two1; rx = nx; ry = 0; }
    else { xs = X.at(0); xi = 1; rx = nx - 1; ys = t0m; ry = ny; }
    uint32_t last = fb(-1.f);
    const uint32_t n_loop = nx + ny + 1;
    for (uint32_t it = 0; it < n_loop; ++it) {
        float v;
        if (xs <= ys) {
            v = xs;
            if (rx > 0) { xs = X.at(xi++); rx--; } else { xs = two; }
        } else {
            v = ys;
            if (ry > 0) { ys = Y.at(yi++); ry--; } else { ys = two1; }
        }
        uint32_t o = fb(v);
        if ((o & 0xFFFFFFFCu) == (last & 0xFFFFFFFCu)) {
            o |= last;
            out[it - 1].y = (int)o;
        }
        out[it] = make_int2((int)r.c, (int)o);
        last = o;
    }
}

// Short and medium pieces (nx + ny + 1 < 128): one thread solves both sides and replays
// the slot walk as it goes, each slot refilled by the next cut of its side -- the same
// sequence walk_piece reads from the stored chains, without storing them.  A step's lanes
// take cuts of both sides in one solve, in a loop that stays rolled: with a solve per side,
// unrolled 16 times, the kernel's 80 KB of code did not fit the instruction cache and a
// 64x64 drawing's k_chains took 153 us for 89.  The output is
// staged: every lane walks kStageSteps entries of its piece into an LDS column, then the
// wave writes the chunk out 16 lanes to a piece, so each piece's run of up to 128 bytes
// goes out in one store instead of one 8-byte store a step (lines left partly written by
// 64 pieces at once were evicted and written back several times: 1.16 GB written a frame
// for 0.42 GB of ts on the 2048x2048 20k-path scene, 0.58 GB now).  A flag merge into an
// entry already written out (equal t's across a chunk boundary, rare) waits for the
// chunk's stores and then updates that entry in memory.
constexpr int kStageSteps = 16;

__device__ __forceinline__ void walk_pieces_staged(PieceSetup &p, bool live, int2 *ts, uint32_t *buf) {
    const int lane = threadIdx.x & 63;
    const uint32_t nx = live ? p.nx : 0u, ny = live ? p.ny : 0u;
    const uint32_t n_loop = live ? nx + ny + 1 : 0u;
    const uint32_t base = live ? p.base : 0u, curve = live ? p.c : 0u;
    const float two = 2.f, two1 = bf(fb(2.f) | 1u);
    float xs = two, ys = two1;
    uint32_t rx = 0, ry = 0;
    float ccx = p.sx.cc, ccy = p.sy.cc;
    const int type = p.sx.type;
    const float w = p.sx.w, t1m = p.sx.t1m;
    if (live) {
        if (nx == 0) { xs = two; ys = p.t0m; rx = 0; ry = ny; }
        else if (ny == 0) { xs = p.t0m; ys = two1; rx = nx; ry = 0; }
        else { xs = p.sx.next(); ccx = p.sx.cc; rx = nx - 1; ys = p.t0m; ry = ny; }
    }
    const uint32_t nmax = (uint32_t)wave_reduce((int)n_loop, 0, OpMaxU());
    uint32_t last = fb(-1.f);
    for (uint32_t it0 = 0; it0 < nmax; it0 += kStageSteps) {
#pragma unroll 1
        for (int j = 0; j < kStageSteps; ++j) {
            const uint32_t it = it0 + j;
            if (it < n_loop) {
                // the slot taken is refilled by its side's next cut, solved from the t just
                // taken; the lanes of both sides share one solve
                const bool tx = xs <= ys;
                const float v = tx ? xs : ys;
                float nv = tx ? two : two1;
                if ((tx ? rx : ry) > 0) {
                    const float t = solve_cut(type, w, tx ? p.sx.a0 : p.sy.a0, tx ? p.sx.a1 : p.sy.a1,
                                              tx ? p.sx.a2 : p.sy.a2, tx ? p.sx.a3 : p.sy.a3, tx ? ccx : ccy, v, t1m);
                    nv = bf((fb(t) & 0xFFFFFFFCu) | (tx ? 0u : 1u));
                    if (tx) { ccx += p.sx.dd; rx--; } else { ccy += p.sy.dd; ry--; }
                }
                xs = tx ? nv : xs;
                ys = tx ? ys : nv;
                uint32_t o = fb(v);
                if ((o & 0xFFFFFFFCu) == (last & 0xFFFFFFFCu)) {
                    o |= last;
                    if (j > 0) {
                        buf[(j - 1) * 64 + lane] = o;
                    } else {
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // the chunk's stores first
                        ts[base + it - 1].y = (int)o;
                    }
                }
                buf[j * 64 + lane] = o;
                last = o;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 4
        for (int k = 0; k < 16; ++k) {
            const int L = 4 * k + (lane >> 4), j = lane & 15;
            const uint32_t nL = (uint32_t)__shfl((int)n_loop, L, 64);
            const uint32_t bL = (uint32_t)__shfl((int)base, L, 64), cL = (uint32_t)__shfl((int)curve, L, 64);
            if (it0 + j < nL) ts[bL + it0 + j] = make_int2((int)cL, (int)buf[j * 64 + L]);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
}

// Intersection pass 1.  Blocks [0, wide_blocks) solve the first cnt[wide_at] chains, cubic
// ones, with several lanes each; the next chain_blocks solve the other listed chains
// of long pieces, longest first; the blocks after them each take 256 short pieces and walk
// them while solving, so the short pieces fill the GPU while the long chains run.  (The word's
// place is an argument: with it written in, the kernel's code came out differently and 1 % slower,
// 254 us for 250 on 3000 mixed paths of 1279x719.)
__global__ void __launch_bounds__(256) k_chains(SceneDev sc, const float4 *__restrict__ crec, const uint4 *__restrict__ clist,
                                                 const uint4 *__restrict__ plist, const uint32_t *__restrict__ cnt,
                                                 uint32_t wide_blocks, int wide_at, uint32_t chain_blocks, int W, int H,
                                                 float *chain_t, int2 *ts) {
    if (blockIdx.x < wide_blocks) {
        wide_chains(sc, crec, clist, cnt[wide_at], wide_blocks, W, H, chain_t);
        return;
    }
    const uint32_t blk = blockIdx.x - wide_blocks;
    if (blk < chain_blocks) {
        // the chains after those of the wide blocks
        const uint32_t i = blk * blockDim.x + threadIdx.x + cnt[wide_at];
        if (i >= chain_total(cnt)) return;
        solve_chain(sc, crec, clist[i], W, H, chain_t);
        return;
    }
    __shared__ uint32_t stage[4][kStageSteps * 64];
    const uint32_t g = (blk - chain_blocks) * blockDim.x + threadIdx.x;
    const uint32_t nlong = cnt[kLongPieceClass];
    const bool live = g < cnt[kListPre + kListClasses] - nlong;
    if (!__ballot(live)) return;  // whole wave past the list
    PieceSetup p;
    if (live) {
        const uint4 e = plist[nlong + g];
        p = piece_setup(sc, crec, e.x >> 3, (int)(e.x & 7u), e, W, H);
    }
    walk_pieces_staged(p, live, ts, stage[threadIdx.x >> 6]);
}

// Long pieces: one two-wave block per piece merges in parallel.  The x chain X and the y
// stream B = [piece start, Y...] are each sorted except that B's start may exceed Y[0]
// by flag bits alone; with B ordered by its running maximum the walk is a stable merge
// (x first on ties): X[i] lands at i + #{B keys < X[i]}, B[j] at j + #{X <= key(B[j])}.
// Runs of equal t then take the OR of their flags up to the next entry of the run.
constexpr int kMergeCap = 1024;
// two waves a piece: the 12 KB window holds a 64-thread block to about three waves per SIMD;
// 128 threads take the headline scene's merge from 258 to 198 us (256: 229 us)
constexpr uint32_t kMergeThreads = 128;

__global__ void __launch_bounds__(kMergeThreads) k_merge_long(const float4 *__restrict__ crec, const float *__restrict__ chain_t,
                                                   const uint4 *__restrict__ plist, const uint32_t *__restrict__ counts,
                                                   int2 *ts) {
    __shared__ float sa[kMergeCap], sb[kMergeCap];
    __shared__ uint32_t sm[kMergeCap];
    const int lane = threadIdx.x;
    const uint32_t n0 = counts[0];
    for (uint32_t g = blockIdx.x; g < n0; g += gridDim.x) {
        const PieceRef r = piece_ref(crec, plist[g]);
        const uint32_t nx = r.nx, ny = r.ny, n = nx + ny + 1;
        if (n > (uint32_t)kMergeCap) {
            // an over-long piece: the walk itself
            if (lane == 0) walk_piece(r, chain_t, ts);
            continue;
        }
        const float *X = chain_t + r.base;
        const float *Y = X + nx;
        if (nx == 0 || ny == 0) {
            // one stream: the piece start, then that chain in order
            const float *Z = nx == 0 ? Y : X;
            for (uint32_t p = lane; p < n; p += kMergeThreads) sm[p] = p == 0 ? fb(r.t0m) : fb(Z[p - 1]);
        } else {
        for (uint32_t i = lane; i < nx; i += kMergeThreads) sa[i] = X[i];
        for (uint32_t j = lane; j <= ny; j += kMergeThreads) sb[j] = j == 0 ? r.t0m : Y[j - 1];
        __syncthreads();
        // running-maximum key of B[j]: max(t0m, Y[j-1]) for j >= 1 (Y is sorted)
        auto bkey = [&](uint32_t j) { return j == 0 ? sb[0] : fmaxf(sb[0], sb[j]); };
        // merge path: each lane merges one contiguous run of outputs [p0, p1), starting
        // from the number of X entries among the first p0 outputs (the first i with
        // X[i] > key(B[p0 - i - 1]), found by binary search)
        const uint32_t nb = ny + 1, seg = (n + kMergeThreads - 1) / kMergeThreads;
        const uint32_t p0 = tmin(n, (uint32_t)lane * seg), p1 = tmin(n, p0 + seg);
        if (p0 < p1) {
            uint32_t lo = p0 > nb ? p0 - nb : 0u, hi = tmin(p0, nx);
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (sa[mid] <= bkey(p0 - mid - 1)) lo = mid + 1; else hi = mid;
            }
            uint32_t i = lo, j = p0 - lo;
            float xv = i < nx ? sa[i] : 0.f, bk = j < nb ? bkey(j) : 0.f;
            for (uint32_t p = p0; p < p1; ++p) {
                const bool takex = i < nx && (j >= nb || xv <= bk);
                if (takex) {
                    sm[p] = fb(xv);
                    ++i;
                    if (i < nx) xv = sa[i];
                } else {
                    sm[p] = fb(sb[j]);
                    ++j;
                    if (j < nb) bk = bkey(j);
                }
            }
        }
        }
        __syncthreads();
        int2 *out = ts + r.base;
        for (uint32_t p = lane; p < n; p += kMergeThreads) {
            const uint32_t v = sm[p], mk = v & 0xFFFFFFFCu;
            uint32_t acc = v;
            for (uint32_t q = p; q > 0 && (sm[q - 1] & 0xFFFFFFFCu) == mk; --q) acc |= sm[q - 1];
            if (p + 1 < n && (sm[p + 1] & 0xFFFFFFFCu) == mk) acc |= sm[p + 1];
            out[p] = make_int2((int)r.c, (int)acc);
        }
        __syncthreads();
    }
}

}  // namespace

// two arrays' tile totals
size_t scan_tmp_elems_needed(size_t n) { return 2 * ((n + kScanTile - 1) / kScanTile + 1); }

void scan_exclusive_u32(const uint32_t *in, uint32_t *out, size_t n, uint32_t *tmp, hipStream_t s) {
    scan_launch(ScanArrays{{in, nullptr}}, 1, ScanOut{{out, nullptr}, {tmp, nullptr}}, n, s);
}

void scan2_exclusive_u32(const uint32_t *in0, uint32_t *out0, const uint32_t *in1, uint32_t *out1, size_t n, uint32_t *tmp,
                         hipStream_t s) {
    scan_launch(ScanArrays{{in0, in1}}, 2, ScanOut{{out0, out1}, {tmp, tmp + scan_tmp_elems_needed(n) / 2}}, n, s);
}

void launch_path_buckets(const SceneDev &sc, Frame &f, hipStream_t s) {
    scan_launch(ScanPathBuckets{f.prow}, 1, ScanOut{{f.pbase, nullptr}, {f.scan_tmp, nullptr}}, sc.P, s);
}

void launch_sizes(const SceneDev &sc, const Frame &f, uint32_t *host, hipStream_t s) {
    hipLaunchKernelGGL(k_sizes, dim3(1), dim3(64), 0, s, (const uint32_t *)f.coff + sc.C, (const uint32_t *)f.choff + sc.C,
                       (const uint32_t *)f.pbase + sc.P, host);
}

void launch_fill_u32(uint32_t *p, uint32_t v, size_t n, hipStream_t s) {
    if (!n) return;
    hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, v, n);
}
void launch_valu_probe(int blocks, int iters, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_valu_probe, dim3(blocks), dim3(256), 0, s, iters, 0.5f, out);
}

void launch_fill_u8(uint8_t *p, uint8_t v, size_t n, hipStream_t s) {
    if (!n) return;
    hipLaunchKernelGGL(k_fill_u8, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, v, n);
}

void launch_fill_rows_u8(uint8_t *p, uint8_t v, size_t row_bytes, size_t pitch, size_t rows, hipStream_t s) {
    const size_t n = row_bytes * rows;
    if (!n) return;
    hipLaunchKernelGGL(k_fill_rows_u8, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, v, row_bytes, pitch, n);
}

void launch_frame_init(const SceneDev &sc, Frame &f, hipStream_t s) {
    hipLaunchKernelGGL(k_frame_init, dim3(std::max(1u, blocks_for(sc.P, 256))), dim3(256), 0, s, sc.P, f.pflags, f.prow, f.big_count);
}

void launch_transform(const SceneDev &sc, Frame &f, hipStream_t s) {
    if (!sc.V) return;
    Mat4 M;
    for (int i = 0; i < 16; ++i) M.m[i] = f.m[i];
    hipLaunchKernelGGL(k_transform, dim3(blocks_for(sc.V, 256)), dim3(256), 0, s, sc.V, sc.vtx, sc.vpath, sc.pcanvas, M,
                       f.W, f.H, f.tvtx, f.pflags);
}

void launch_monotone(const SceneDev &sc, Frame &f, hipStream_t s) {
    if (!sc.C) return;
    hipLaunchKernelGGL(k_monotone, dim3(blocks_for(sc.C, 256)), dim3(256), 0, s, sc, (const float2 *)f.tvtx,
                       (const uint32_t *)f.pflags, f.W, f.H, f.crec, f.cfrag, f.pcnt, f.nchain, f.prow);
}

void launch_intersect(const SceneDev &sc, Frame &f, hipStream_t s) {
    if (!sc.C) return;
    uint32_t *cnt = f.lcount;
    // Cubic chains of the first length bins take several lanes each (wide_chains): one
    // lane's 1.5 us a cut makes the longest chains the pass's time in frames of every size, but
    // the lanes cost up to 20 times the issue slots, so the more cuts a frame has, the fewer
    // chains pay.  Pieces of cubic_min cuts are listed as chains; shorter ones are walked by one
    // lane.  Intersection stage, one lane a chain / the rule, us: 3.5 k cuts 111 / 67, 0.45 M
    // 415 / 219, 2.1 M 515 / 385, 2.9 M 528 / 296, 5 M 483 / 300, 6.2 M 712 / 380, 12.8 M
    // 782 / 484, 26 M 840 / 566, 51 M 985 / 719.  Neighbouring settings at each limit: 5 M with
    // three bins 341, 6.2 M with four 387 and two 458, 12.8 M with four 570, 26 M with three 698,
    // 51 M with three 1115; 2.1 M with 128-cut pieces and four bins 439.
    // The bins end earlier where their chains are too many (the loads): the lanes' work then
    // lasts longer than the longest chain would on one lane.  Stage at the loads times 1/2, 1,
    // 4/3, 2 and without a limit, us: 4000 curves of 500 cuts (6.4 M cuts) 745, 746, 746, 1150,
    // 1139, a lane each 742; 3000 drawn chains seen at 1:4 (24 M) 1521, 1517, 1497, 1515, 6803,
    // a lane each 1501; 3800 curves of 60 cuts a side (0.9 M) 107, 107, 148, 144, 145; where
    // the lanes pay, 1000 drawn chains of 1000x1000 (4.4 M) 564, 555, 592, 776, 781, a lane
    // each 797, and the 51 M above 857, 720, 720, 720, 719.
    const struct { int64_t cuts; uint32_t cubic_min; WideRule wide; uint32_t blocks; } rule[] = {
        {1 << 18, 24u, {kLenBins, 6144u}, 2048u}, {1 << 21, 64u, {kLenBins, 6144u}, 2048u},
        {5 << 20, kLongPiece, {4, 3072u}, 512u},  {1 << 24, kLongPiece, {3, 2304u}, 256u},
        {INT64_MAX, kLongPiece, {2, 2304u}, 256u}};
    int at = 0;
    while (f.F > rule[at].cuts) ++at;
    const uint32_t cubic_min = rule[at].cubic_min;
    const WideRule wide = rule[at].wide;
    // One block, for up to 1024 curves, counts and places by itself: 9.6 us for the two launches'
    // 13.6 with 91 curves, but with 1591 25 for 21.  More blocks leave their counts in the curves'
    // fragment counts, which their scan was the last to read: 101 words a block for a word a curve,
    // so they fit however few cuts the frame has.  (With the blocks cut down to the chains' t
    // array, a view of 154 cuts of a sheet of 6.2 M curves took 5.7 ms for the stage, now 37 us.)
    const dim3 bl(kChainListThreads);
    uint32_t nb = std::min<uint32_t>(blocks_for(sc.C, kChainListThreads), kListBlocks);
    const uint32_t per = blocks_for(blocks_for(sc.C, kChainListThreads), nb) * kChainListThreads;
    nb = blocks_for(sc.C, per);
    static_assert(2 * kListClasses <= kChainListThreads, "the block counts exceed the curves' words");
    uint32_t *blk = f.cfrag;
    if (nb == 1) {
        hipLaunchKernelGGL(k_list_place<true>, dim3(1), bl, 0, s, sc, sc.C, per, (const uint32_t *)f.nchain,
                           (const uint32_t *)f.pcnt, (const uint32_t *)f.coff, cubic_min, wide, (const uint32_t *)nullptr, cnt,
                           f.chains, f.plist);
    } else {
        hipLaunchKernelGGL(k_list_count, dim3(nb), bl, 0, s, sc, sc.C, per, (const uint32_t *)f.nchain,
                           (const uint32_t *)f.pcnt, cubic_min, blk);
        hipLaunchKernelGGL(k_list_place<false>, dim3(nb), bl, 0, s, sc, sc.C, per, (const uint32_t *)f.nchain,
                           (const uint32_t *)f.pcnt, (const uint32_t *)f.coff, cubic_min, wide, (const uint32_t *)blk, cnt,
                           f.chains, f.plist);
    }
    // chain blocks: enough for every chain; piece blocks: enough for every piece
    const uint32_t npieces = (uint32_t)(f.NCH / 2);
    const uint32_t chain_blocks = blocks_for(f.NCH, 256), piece_blocks = blocks_for(npieces, 256);
    const uint32_t wide_blocks = std::min<uint32_t>(rule[at].blocks, blocks_for(f.NCH, 4));
    if (f.NCH)
        hipLaunchKernelGGL(k_chains, dim3(wide_blocks + chain_blocks + piece_blocks), dim3(256), 0, s, sc, (const float4 *)f.crec,
                           (const uint4 *)f.chains, (const uint4 *)f.plist,
                           (const uint32_t *)cnt, wide_blocks, kListWide, chain_blocks, f.W, f.H, f.chain_t, f.ts);
    // one block per long piece up to 32768 blocks: the pieces' sizes vary widely, and
    // blocks that find no piece exit at once
    if (npieces)
        hipLaunchKernelGGL(k_merge_long, dim3(npieces < 32768u ? npieces : 32768u), dim3(kMergeThreads), 0, s,
                           (const float4 *)f.crec, (const float *)f.chain_t, (const uint4 *)f.plist,
                           (const uint32_t *)(cnt + kLongPieceClass), f.ts);
}

}  // namespace sl
