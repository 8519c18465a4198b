// sl_diff.hip -- differentiable mode: a forward renderer with continuous coverage and its
// hand-written adjoint (the reference has no such mode).
//
// Model.  A pixel row y holds S sample rows at y + (s + 1/2)/S.  Along each sample row the
// fill indicator of a path (nonzero / even-odd over the signed crossings of the row) is
// integrated exactly over every pixel's [x, x+1), so coverage is a box filter of S rows,
// continuous in the control points:
//     cov_p(x, y) = (1/S) * sum_s |{u in [x, x+1) : fill_p(u, y_s)}|
// and the image is the renderer's src-over onto white, in path order, unquantised:
//     a = paint_a * cov;  rgb = paint * a + rgb * (1 - a);  A = a * a + A * (1 - a).
//
// Forward: crossings of every y-monotone curve piece with the sample rows (half-open rule
// ymin <= y_s < ymax, bisection on t), bucketed by (path, sample row) and sorted by x; the
// fill change at each crossing; coverage per (path, pixel row) by one wavefront; the
// compositing chain per pixel (the colour before each path is kept for the adjoint).
// Adjoint: the chain reversed per pixel gives d/d paint and d/d cov; then every crossing
// with a fill change contributes d cov / d x_i = (fill left - fill right) / S in its pixel,
// and x_i = Bx(t*) with By(t*) = y_s moves with the control points as
//     d x_i / d Pk.x = b_k(t*),   d x_i / d Pk.y = -Bx'(t*) / By'(t*) * b_k(t*).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "../../include/scanline.h"
#include "sl_device.h"
#include "sl_internal.h"

namespace {

template <class T> __device__ __forceinline__ T tmn(T a, T b) { return a < b ? a : b; }
template <class T> __device__ __forceinline__ T tmx(T a, T b) { return a > b ? a : b; }

struct DSeg {
    int type;
    float x[4], y[4];
};

__device__ __forceinline__ DSeg load_seg(const float2 *__restrict__ pts, const uint32_t *__restrict__ cvpos,
                                         const uint8_t *__restrict__ ctype, uint32_t c) {
    DSeg g;
    g.type = ctype[c];
    const int nv = g.type & 7;
    const uint32_t v0 = cvpos[c];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float2 p = pts[v0 + (uint32_t)(k < nv ? k : nv - 1)];
        g.x[k] = p.x;
        g.y[k] = p.y;
    }
    return g;
}

__device__ __forceinline__ float bez(int type, const float *p, float t) {
    const float s = 1.f - t;
    if (type == 2) return s * p[0] + t * p[1];
    if (type == 3) return s * s * p[0] + 2.f * s * t * p[1] + t * t * p[2];
    return s * s * s * p[0] + 3.f * s * s * t * p[1] + 3.f * s * t * t * p[2] + t * t * t * p[3];
}

__device__ __forceinline__ float dbez(int type, const float *p, float t) {
    const float s = 1.f - t;
    if (type == 2) return p[1] - p[0];
    if (type == 3) return 2.f * (s * (p[1] - p[0]) + t * (p[2] - p[1]));
    return 3.f * (s * s * (p[1] - p[0]) + 2.f * s * t * (p[2] - p[1]) + t * t * (p[3] - p[2]));
}

__device__ __forceinline__ void basis(int type, float t, float *b) {
    const float s = 1.f - t;
    b[0] = b[1] = b[2] = b[3] = 0.f;
    if (type == 2) {
        b[0] = s;
        b[1] = t;
    } else if (type == 3) {
        b[0] = s * s;
        b[1] = 2.f * s * t;
        b[2] = t * t;
    } else {
        b[0] = s * s * s;
        b[1] = 3.f * s * s * t;
        b[2] = 3.f * s * t * t;
        b[3] = t * t * t;
    }
}

// t of the y-extrema inside (0, 1), ascending; the piece boundaries are {0, these, 1}
__device__ __forceinline__ int y_extrema(int type, const float *y, float *r) {
    int n = 0;
    if (type == 3) {
        const float den = y[0] - 2.f * y[1] + y[2];
        if (den != 0.f) {
            const float t = (y[0] - y[1]) / den;
            if (t > 0.f && t < 1.f) r[n++] = t;
        }
    } else if (type == 4) {
        const float a = -y[0] + 3.f * y[1] - 3.f * y[2] + y[3];
        const float b = 2.f * (y[0] - 2.f * y[1] + y[2]);
        const float c = y[1] - y[0];
        if (a == 0.f) {
            if (b != 0.f) {
                const float t = -c / b;
                if (t > 0.f && t < 1.f) r[n++] = t;
            }
        } else {
            const float disc = b * b - 4.f * a * c;
            if (disc > 0.f) {
                const float sq = sqrtf(disc);
                float t0 = (-b - sq) / (2.f * a), t1 = (-b + sq) / (2.f * a);
                if (t0 > t1) {
                    const float tt = t0;
                    t0 = t1;
                    t1 = tt;
                }
                if (t0 > 0.f && t0 < 1.f) r[n++] = t0;
                if (t1 > 0.f && t1 < 1.f && t1 != t0) r[n++] = t1;
            }
        }
    }
    return n;
}

// first sample row j with (j + 1/2)/S >= y, clamped to [-1, J + 1] (NaN -> -1)
__device__ __forceinline__ long first_row(float y, int S, long J) {
    float v = ceilf(y * (float)S - 0.5f);
    if (!(v >= -1.f)) v = -1.f;
    if (v > (float)(J + 1)) v = (float)(J + 1);
    return (long)v;
}

// Pieces of a segment and their sample-row ranges [ja, jb); returns the piece count.
struct Pieces {
    int n;
    float t[4];
    int ja[3], jb[3], dir[3];
};

__device__ __forceinline__ Pieces pieces(const DSeg &g, int S, long J) {
    Pieces pc;
    float ts[4] = {0.f, 0.f, 0.f, 0.f};
    const int ne = y_extrema(g.type, g.y, ts + 1);
    ts[ne + 1] = 1.f;
    pc.n = ne + 1;
    float yprev = bez(g.type, g.y, 0.f);
    for (int k = 0; k < 4; ++k) pc.t[k] = ts[k];
    for (int k = 0; k < 3; ++k) {
        pc.ja[k] = pc.jb[k] = 0;
        pc.dir[k] = 0;
        if (k > ne) continue;
        const float y0 = yprev, y1 = bez(g.type, g.y, ts[k + 1]);
        yprev = y1;
        if (y0 == y1) continue;
        const float ylo = fminf(y0, y1), yhi = fmaxf(y0, y1);
        const long ja = tmx(first_row(ylo, S, J), 0L), jb = tmn(first_row(yhi, S, J), J);
        if (jb > ja) {
            pc.ja[k] = (int)ja;
            pc.jb[k] = (int)jb;
        }
        pc.dir[k] = y1 > y0 ? 1 : -1;
    }
    return pc;
}

struct DiffDev {
    int W, H, S, P;
    uint32_t C;
    const uint32_t *cvpos, *cpath;
    const uint8_t *ctype, *frule;
};

__global__ void k_d_count(DiffDev D, const float2 *__restrict__ pts, uint32_t *cnt) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= D.C) return;
    const DSeg g = load_seg(pts, D.cvpos, D.ctype, c);
    const Pieces pc = pieces(g, D.S, (long)D.H * D.S);
    uint32_t n = 0;
    for (int k = 0; k < pc.n; ++k) n += (uint32_t)(pc.jb[k] - pc.ja[k]);
    cnt[c] = n;
}

struct Cross {
    float x, t;
    uint32_t curve;
    uint32_t row_dir;  // sample row << 1 | (dir > 0)
};

__global__ void k_d_cross(DiffDev D, const float2 *__restrict__ pts, const uint32_t *__restrict__ off, uint32_t NX,
                          Cross *xs, uint32_t *key, uint32_t *rank, uint32_t *bcount) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NX) return;
    // the curve holding crossing i: last c with off[c] <= i
    uint32_t lo = 0, hi = D.C - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid; else hi = mid - 1;
    }
    const uint32_t c = lo;
    const DSeg g = load_seg(pts, D.cvpos, D.ctype, c);
    const Pieces pc = pieces(g, D.S, (long)D.H * D.S);
    uint32_t r = i - off[c];
    int k = 0;
    for (; k < pc.n - 1; ++k) {
        const uint32_t m = (uint32_t)(pc.jb[k] - pc.ja[k]);
        if (r < m) break;
        r -= m;
    }
    const int j = pc.ja[k] + (int)r, dir = pc.dir[k];
    const float ys = ((float)j + 0.5f) / (float)D.S;
    float tl = dir > 0 ? pc.t[k] : pc.t[k + 1], th = dir > 0 ? pc.t[k + 1] : pc.t[k];
    for (int it = 0; it < 32; ++it) {
        const float mid = 0.5f * (tl + th);
        if (bez(g.type, g.y, mid) < ys) tl = mid; else th = mid;
    }
    const float t = 0.5f * (tl + th);
    Cross o;
    o.x = bez(g.type, g.x, t);
    o.t = t;
    o.curve = c;
    o.row_dir = ((uint32_t)j << 1) | (dir > 0 ? 1u : 0u);
    xs[i] = o;
    const uint32_t b = D.cpath[c] * (uint32_t)(D.H * D.S) + (uint32_t)j;
    key[i] = b;
    rank[i] = atomicAdd(&bcount[b], 1u);  // the crossing's place in its bucket (any order)
}

__global__ void k_d_scatter(uint32_t NX, const uint32_t *__restrict__ key, const uint32_t *__restrict__ rank,
                            const uint32_t *__restrict__ boff, uint32_t *order) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < NX) order[boff[key[i]] + rank[i]] = i;
}

__device__ __forceinline__ bool filled(int rule, int w) { return rule ? (w & 1) != 0 : w != 0; }

// Order of a bucket's crossings: (x, curve, t, index), x as an unsigned key that orders like
// the float (every NaN last, -0 and +0 equal), so the order is total whatever the values.
__device__ __forceinline__ uint32_t order_key(float x) {
    if (x != x) return 0xFFFFFFFFu;
    const uint32_t u = __float_as_uint(x + 0.f);
    return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ bool comes_before(uint32_t ax, uint32_t ac, uint32_t at, uint32_t ai, uint32_t bx, uint32_t bc,
                                             uint32_t bt, uint32_t bi) {
    if (ax != bx) return ax < bx;
    if (ac != bc) return ac < bc;
    if (at != bt) return at < bt;  // t >= 0: the bits order like the values
    return ai < bi;
}

__device__ __forceinline__ int wave_scan_add(int x) { return sl::dev::dpp_scan(x, 0, sl::dev::OpAdd()); }

// Fill changes and coverage, one wavefront per (path, pixel row): the row's sample rows are
// neighbouring buckets, so their crossings are one run of `order`.  A lane takes a crossing:
// its winding is the sum of the directions of the bucket's crossings before it (no sorted
// order is stored), the fill change follows, and the area right of the crossing goes into
// the row's pixels as a second difference -- turn (p + 1 - u) at its pixel p, the rest of
// turn at p + 1 -- so that a running sum over x gives every pixel's coverage.  Right of a
// bucket's last crossing nothing is filled, also where its winding does not return to zero
// (open contours: points that moved one segment at a time).  The sums are
// 32-bit fixed point, 2^-25 of a sample row: the atomics' order does not matter, the two
// parts of a crossing add to exactly one, and a pixel's sum (at most 64 rows) fits 32 bits.
// From x = 1/4 on a float's fraction is a multiple of 2^-25, so the sums are exact; what a
// crossing left of that has below, only column 0 feels, and the lanes keep it in registers in
// units of 2^-56 (slivers of 2^-32 of a pixel keep a float's precision).
// A crossing costs one pass over its bucket and two LDS adds, where integrating every
// interval over every pixel column cost each column a pass over the whole row's crossings.
// 861 k crossings (64 paths at 256x256, 16 rows): 26 us, where sorting the buckets and the
// column passes took 35 and 237 us.
constexpr int kFillStage = 128;   // crossings of a row staged in LDS (more are read from memory)
constexpr int kFillPixels = 512;  // pixel columns of one pass over a row
constexpr float kAreaScale = 33554432.f;  // 2^25
constexpr float kRestScale = 2147483648.f;  // 2^31: the rest's units in one of the area's

// What k_d_fill keeps of a crossing: the fill's change (left - right, by the windings) for the
// adjoint, and the coverage's (right - left, with nothing after the last crossing).
__device__ __forceinline__ uint8_t turn_code(int change, int turn) { return (uint8_t)((change + 1) | ((turn + 1) << 2)); }
__device__ __forceinline__ int code_change(uint8_t c) { return (int)(c & 3) - 1; }
__device__ __forceinline__ int code_turn(uint8_t c) { return (int)(c >> 2) - 1; }

__global__ void __launch_bounds__(256) k_d_fill(DiffDev D, const uint32_t *__restrict__ boff,
                                                const uint32_t *__restrict__ order, const Cross *__restrict__ xs,
                                                uint8_t *df, float *__restrict__ cov) {
    __shared__ uint4 s_cr[4][kFillStage];       // {x key, curve, t bits, index << 1 | dir}
    __shared__ uint32_t s_sum[4][kFillPixels];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t wid = (int64_t)blockIdx.x * 4 + wv;
    const bool live = wid < (int64_t)D.P * D.H;
    const int p = live ? (int)(wid / D.H) : 0, y = live ? (int)(wid - (int64_t)p * D.H) : 0;
    const int rule = D.frule[p];
    const uint32_t b0 = (uint32_t)p * (uint32_t)(D.H * D.S) + (uint32_t)(y * D.S);
    const uint32_t r0 = live ? boff[b0] : 0u, n = live ? boff[b0 + D.S] - r0 : 0u;
    uint4 *cr = s_cr[wv];
    uint32_t *sum = s_sum[wv];
    const uint32_t nst = tmn(n, (uint32_t)kFillStage);
    auto load = [&](uint32_t k) {
        const uint32_t i = order[r0 + k];
        const Cross c = xs[i];
        return make_uint4(order_key(c.x), c.curve, __float_as_uint(c.t), (i << 1) | (c.row_dir & 1u));
    };
    for (uint32_t k = lane; k < nst; k += 64) cr[k] = load(k);
    __syncthreads();
    const float Wf = (float)D.W;
    float *row = cov + ((size_t)p * D.H + y) * D.W;
    for (int x0 = 0; x0 < D.W; x0 += kFillPixels) {
        for (int k = lane; k < kFillPixels; k += 64) sum[k] = 0u;
        __syncthreads();
        uint32_t carry = 0u;  // what lies left of this pass's columns
        long long rest = 0;   // what column 0 has below the sums' unit, taken off
        for (uint32_t k = lane; k < n; k += 64) {
            const uint32_t i = order[r0 + k];
            const Cross c = xs[i];
            int turn;
            if (x0 == 0) {
                const uint32_t b = b0 + (c.row_dir >> 1) - (uint32_t)(y * D.S);
                const uint32_t a0 = boff[b] - r0, a1 = boff[b + 1] - r0;
                const uint32_t kx = order_key(c.x), kt = __float_as_uint(c.t);
                int w = 0;
                uint32_t left = a1 - a0 - 1u;  // crossings that come after this one
                for (uint32_t m = a0; m < a1; ++m) {
                    const uint4 q = m < nst ? cr[m] : load(m);
                    if (comes_before(q.x, q.y, q.z, q.w >> 1, kx, c.curve, kt, i & 0x7FFFFFFFu)) {
                        w += (q.w & 1u) ? 1 : -1;
                        --left;
                    }
                }
                const int d = (c.row_dir & 1u) ? 1 : -1;
                const int in0 = filled(rule, w) ? 1 : 0, in1 = filled(rule, w + d) ? 1 : 0;
                turn = (left ? in1 : 0) - in0;
                df[i] = turn_code(in0 - in1, turn);
            } else {
                turn = code_turn(df[i]);  // written by this lane in the first pass
            }
            if (!turn) continue;
            // a crossing without a position, last in the order, lies at the right edge: the
            // positions then never decrease along the order, and a row fills no pixel twice
            const float u = c.x < Wf ? fmaxf(c.x, 0.f) : Wf;
            const int px = (int)floorf(u);
            const float at = (u - (float)px) * kAreaScale, part = rintf(at);  // exact but for the rounding
            if (px == 0) rest += turn * __float2ll_rn((at - part) * kRestScale);
            const int v = (int)kAreaScale - (int)part;
            const uint32_t va = (uint32_t)(turn * v), vb = (uint32_t)(turn * (int)part);
            const int q = px - x0;
            if (q < 0) carry += va;
            else if (q < kFillPixels) atomicAdd(&sum[q], va);
            if (q + 1 < 0) carry += vb;
            else if (q + 1 < kFillPixels) atomicAdd(&sum[q + 1], vb);
        }
        __syncthreads();
        carry = (uint32_t)__builtin_amdgcn_readlane(wave_scan_add((int)carry), 63);
        const int xe = tmn(D.W - x0, kFillPixels);
        const bool fine = x0 == 0 && __ballot(rest != 0);
        if (fine) {
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) rest += __shfl_xor(rest, d, 64);
        }
        for (int k0 = 0; k0 < xe; k0 += 64) {
            const uint32_t s = (uint32_t)wave_scan_add((int)sum[k0 + lane]) + carry;
            carry = (uint32_t)__builtin_amdgcn_readlane((int)s, 63);
            float c = (float)s * (1.f / kAreaScale);
            if (fine && k0 + lane == 0)  // at most 2^62
                c = (float)((long long)((unsigned long long)s << 31) - rest) * (1.f / kAreaScale / kRestScale);
            if (live && k0 + lane < xe) row[x0 + k0 + lane] = c / (float)D.S;
        }
        __syncthreads();
    }
}

__global__ void k_d_composite(DiffDev D, const float *__restrict__ cov, const float4 *__restrict__ col,
                              float4 *__restrict__ pre, float4 *__restrict__ img) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t NP = (int64_t)D.W * D.H;
    if (i >= NP) return;
    float I0 = 1.f, I1 = 1.f, I2 = 1.f, I3 = 1.f;
    for (int p = 0; p < D.P; ++p) {
        if (pre) pre[(size_t)p * NP + i] = make_float4(I0, I1, I2, I3);
        const float4 c = col[p];
        const float a = c.w * cov[(size_t)p * NP + i];
        const float oma = 1.f - a;
        I0 = c.x * a + I0 * oma;
        I1 = c.y * a + I1 * oma;
        I2 = c.z * a + I2 * oma;
        I3 = a * a + I3 * oma;
    }
    img[i] = make_float4(I0, I1, I2, I3);
}

// Gradient sums are accumulated in 64-bit fixed point, 2^-32 units: each contribution is
// rounded once (to nearest) and added with an integer atomic.  Integer addition is
// associative, so the sums do not depend on the order the atomics land in and every run
// gives the same bits; a float atomicAdd's result depends on that order.  Contributions
// are clamped to |v| <= 2^30 and the sums stay far inside the int64 range for any
// gradient image of moderate size.
constexpr double kFixScale = 4294967296.0;  // 2^32

__global__ void k_d_unfix(const long long *__restrict__ acc, float *__restrict__ out, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = (float)((double)acc[i] * (1.0 / kFixScale));
}

// The sum of v over the wave, in every lane: DPP row shifts and broadcasts (no LDS trips).
__device__ __forceinline__ float wave_sum(float v) {
#define SL_STEP(ctrl, mask) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, mask, 0xf, false))
    SL_STEP(0x111, 0xf);
    SL_STEP(0x112, 0xf);
    SL_STEP(0x114, 0xf);
    SL_STEP(0x118, 0xf);
    SL_STEP(0x142, 0xa);
    SL_STEP(0x143, 0xc);
#undef SL_STEP
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ long long fix_of(float v) {
    return __double2ll_rn(fmin(fmax((double)v, -1073741824.0), 1073741824.0) * kFixScale);
}

// Adjoint of the compositing chain, one thread per pixel.  A path's four colour sums are
// reduced over the wave, collected per block in LDS (kBackPaths paths at a time) and added
// to memory once per block; a wave none of whose pixels the path covers has nothing to add.
// 64 paths at 256x256: 31 us (101 MB of colours and coverages, 3.2 TB/s, on one wave per
// SIMD), 47 us without loading a path ahead; one global atomic a wave, path and channel,
// after shuffle reductions, took 111 us.
constexpr int kBackPaths = 256;

__global__ void __launch_bounds__(256) k_d_back_pixels(DiffDev D, const float *__restrict__ cov,
                                                       const float4 *__restrict__ col, const float4 *__restrict__ pre,
                                                       const float4 *__restrict__ gimg, float *__restrict__ gcov,
                                                       unsigned long long *__restrict__ gcol) {
    __shared__ unsigned long long s_acc[4 * kBackPaths];
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t NP = (int64_t)D.W * D.H;
    const bool in = i < NP;
    float4 g = in ? gimg[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p1 = D.P; p1 > 0; p1 -= kBackPaths) {
        const int p0 = tmx(p1 - kBackPaths, 0);
        for (int k = threadIdx.x; k < 4 * (p1 - p0); k += 256) s_acc[k] = 0ull;
        __syncthreads();
        float4 npr = make_float4(0.f, 0.f, 0.f, 0.f);
        float ncv = 0.f;
        if (in) {
            npr = pre[(size_t)(p1 - 1) * NP + i];
            ncv = cov[(size_t)(p1 - 1) * NP + i];
        }
        for (int p = p1 - 1; p >= p0; --p) {
            const float4 c = col[p];
            const float4 pr = npr;
            const float cv = ncv;
            float a = 0.f, da = 0.f;
            if (in && p > p0) {  // the next path's values load during this one's arithmetic
                npr = pre[(size_t)(p - 1) * NP + i];
                ncv = cov[(size_t)(p - 1) * NP + i];
            }
            if (in) {
                a = c.w * cv;
                da = g.x * (c.x - pr.x) + g.y * (c.y - pr.y) + g.z * (c.z - pr.z) + g.w * (2.f * a - pr.w);
                gcov[(size_t)p * NP + i] = da * c.w;
            }
            if (__ballot(cv != 0.f || a != 0.f)) {
                const float s0 = wave_sum(g.x * a), s1 = wave_sum(g.y * a), s2 = wave_sum(g.z * a), s3 = wave_sum(da * cv);
                const float s = lane == 0 ? s0 : (lane == 1 ? s1 : (lane == 2 ? s2 : s3));
                if (lane < 4 && s != 0.f) atomicAdd(&s_acc[4 * (p - p0) + lane], (unsigned long long)fix_of(s));
            }
            const float oma = 1.f - a;
            g.x *= oma;
            g.y *= oma;
            g.z *= oma;
            g.w *= oma;
        }
        __syncthreads();
        for (int k = threadIdx.x; k < 4 * (p1 - p0); k += 256)
            if (s_acc[k]) atomicAdd(&gcol[4 * (size_t)p0 + k], s_acc[k]);
        __syncthreads();
    }
}

// Boundary terms at the crossings, in the order they were found: a curve's crossings are
// neighbours, so a wave takes a curve (blockIdx.x; blockIdx.y of gridDim.y shares of its
// crossings), each lane sums its crossings' fixed-point terms for the curve's points in
// registers, and the wave adds each sum to memory once.  Every term is rounded by itself
// before it is added, as a sum of atomics would have it, so the split does not change the
// result.  861 k crossings of 384 curves: 19 us, bound by the gathers of gcov; one atomic
// per crossing, point and coordinate took 500 us, some 2200 of them meeting at each address.
__global__ void __launch_bounds__(64) k_d_back_cross(DiffDev D, const uint32_t *__restrict__ off,
                                                     const Cross *__restrict__ xs, const uint8_t *__restrict__ df,
                                                     const float2 *__restrict__ pts, const float *__restrict__ gcov,
                                                     unsigned long long *gpts) {
    const uint32_t c = blockIdx.x;
    const uint32_t i0 = off[c], i1 = off[c + 1];
    if (i0 == i1) return;
    const DSeg g = load_seg(pts, D.cvpos, D.ctype, c);
    const size_t NP = (size_t)D.W * D.H;
    const float *gp = gcov + (size_t)D.cpath[c] * NP;
    long long sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const int nv = g.type & 7;
    for (uint32_t i = i0 + blockIdx.y * 64u + threadIdx.x; i < i1; i += 64u * gridDim.y) {
        const int f = code_change(df[i]);
        if (!f) continue;
        const Cross cr = xs[i];
        if (!(cr.x >= 0.f && cr.x < (float)D.W)) continue;
        const int j = (int)(cr.row_dir >> 1), y = j / D.S;
        const int px = (int)floorf(cr.x);
        const float gx = gp[(size_t)y * D.W + px] * (float)f / (float)D.S;
        if (gx == 0.f) continue;
        float b[4];
        basis(g.type, cr.t, b);
        // dx/dy along the curve; near a y-extremum By' -> 0, bounded at |By'| >= 1e-4
        float dyv = dbez(g.type, g.y, cr.t);
        if (fabsf(dyv) < 1e-4f) dyv = dyv < 0.f ? -1e-4f : 1e-4f;
        const float ratio = dbez(g.type, g.x, cr.t) / dyv;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (v < nv) {
                sum[2 * v] += fix_of(gx * b[v]);
                sum[2 * v + 1] += fix_of(-gx * ratio * b[v]);
            }
        }
    }
    const uint32_t v0 = D.cvpos[c];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        long long s = sum[v];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
        if (threadIdx.x == 0 && s && v < 2 * nv) atomicAdd(&gpts[2 * (size_t)v0 + v], (unsigned long long)s);
    }
}

__global__ void k_d_clear(float *p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.f;
}

inline unsigned nblk(int64_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }
// waves a curve's crossings are shared by: about four crossings a lane on the average curve
inline unsigned shares_of(uint32_t NX, uint32_t C) {
    return (unsigned)std::min<size_t>(64, std::max<size_t>(1, NX / ((size_t)C * 256)));
}

struct Buf {
    void *p = nullptr;
    size_t cap = 0;
};

}  // namespace

struct sl_diff {
    int device = 0;
    int W = 0, H = 0, S = 16;
    uint32_t P = 0, C = 0, V = 0;
    Buf cvpos, cpath, ctype, frule;
    Buf cnt, off, xs, key, rank, bcount, boff, order, df, cov, pre, gcov, scan_tmp;
    Buf gfix;  // fixed-point gradient sums: 2V point components, then 4P colour components
    uint32_t NX = 0;
    bool have_pre = false;
    const float *last_points = nullptr, *last_colors = nullptr;
    // the last forward or backward, possibly still running on last_stream
    hipEvent_t done_ev = nullptr;
    hipStream_t last_stream = nullptr;
    bool pending = false;
    std::string err;
};

namespace {

int dfail(sl_diff *d, int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (d) d->err = buf;
    return code;
}

// Forward and backward share the handle's buffers.  Work issued on another stream than
// the last call's waits on the host until that call has finished.
int diff_order(sl_diff *d, hipStream_t s) {
    if (d->pending && s != d->last_stream) {
        if (hipEventSynchronize(d->done_ev) != hipSuccess) return dfail(d, SL_E_HIP, "previous call failed");
        d->pending = false;
    }
    return SL_OK;
}

int diff_issued(sl_diff *d, hipStream_t s) {
    if (!d->done_ev && hipEventCreateWithFlags(&d->done_ev, hipEventDisableTiming) != hipSuccess)
        return dfail(d, SL_E_HIP, "hipEventCreate failed");
    if (hipEventRecord(d->done_ev, s) != hipSuccess) return dfail(d, SL_E_HIP, "hipEventRecord failed");
    d->pending = true;
    d->last_stream = s;
    return SL_OK;
}

int dens(sl_diff *d, Buf &b, size_t bytes) {
    if (bytes == 0) bytes = 16;
    if (b.cap >= bytes) return SL_OK;
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    const size_t want = bytes + bytes / 4;
    if (hipMalloc(&b.p, want) != hipSuccess) {
        b.p = nullptr;
        (void)hipGetLastError();
        return dfail(d, SL_E_OOM, "hipMalloc(%zu) failed", want);
    }
    b.cap = want;
    return SL_OK;
}

template <class T> T *BP(Buf &b) { return (T *)b.p; }

DiffDev dev_view(sl_diff *d) {
    DiffDev D;
    D.W = d->W; D.H = d->H; D.S = d->S; D.P = (int)d->P; D.C = d->C;
    D.cvpos = BP<uint32_t>(d->cvpos); D.cpath = BP<uint32_t>(d->cpath);
    D.ctype = BP<uint8_t>(d->ctype); D.frule = BP<uint8_t>(d->frule);
    return D;
}

}  // namespace

extern "C" {

int sl_diff_create(int device, int width, int height, int sample_rows, uint32_t n_paths, uint32_t n_curves,
                   uint32_t n_vertices, const uint32_t *curve_vertex_pos, const uint8_t *curve_type,
                   const uint32_t *curve_path_id, const uint8_t *fill_rule, sl_diff **out) {
    if (!out || width <= 0 || height <= 0 || sample_rows <= 0 || sample_rows > 64 || n_paths == 0 ||
        n_curves == 0 || !curve_vertex_pos || !curve_type || !curve_path_id || !fill_rule)
        return SL_E_ARG;
    *out = nullptr;
    if ((uint64_t)n_paths * height * sample_rows >= 0xFFFFFFFFull) return SL_E_UNSUPPORTED;
    if ((uint64_t)n_paths * width * height > (1ull << 28)) return SL_E_UNSUPPORTED;
    for (uint32_t c = 0; c < n_curves; ++c) {
        const int t = curve_type[c];
        if (t != SL_CURVE_LINEAR && t != SL_CURVE_QUADRATIC && t != SL_CURVE_CUBIC) return SL_E_UNSUPPORTED;
        if ((uint64_t)curve_vertex_pos[c] + (t & 7) > n_vertices) return SL_E_ARG;
        if (curve_path_id[c] >= n_paths || (c && curve_path_id[c] < curve_path_id[c - 1])) return SL_E_ARG;
    }
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return SL_E_NODEVICE;
    }
    if (device < 0) device = 0;
    if (device >= n || hipSetDevice(device) != hipSuccess) return SL_E_ARG;
    sl_diff *d = new (std::nothrow) sl_diff;
    if (!d) return SL_E_OOM;
    d->device = device;
    d->W = width; d->H = height; d->S = sample_rows;
    d->P = n_paths; d->C = n_curves; d->V = n_vertices;
    int rc;
    if ((rc = dens(d, d->cvpos, (size_t)n_curves * 4)) || (rc = dens(d, d->cpath, (size_t)n_curves * 4)) ||
        (rc = dens(d, d->ctype, n_curves)) || (rc = dens(d, d->frule, n_paths))) {
        sl_diff_destroy(d);
        return rc;
    }
    if (hipMemcpy(d->cvpos.p, curve_vertex_pos, (size_t)n_curves * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d->cpath.p, curve_path_id, (size_t)n_curves * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d->ctype.p, curve_type, n_curves, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d->frule.p, fill_rule, n_paths, hipMemcpyHostToDevice) != hipSuccess) {
        sl_diff_destroy(d);
        return SL_E_HIP;
    }
    *out = d;
    return SL_OK;
}

int sl_diff_destroy(sl_diff *d) {
    if (!d) return SL_OK;
    (void)hipSetDevice(d->device);
    (void)hipDeviceSynchronize();
    Buf *bs[] = {&d->cvpos, &d->cpath, &d->ctype, &d->frule, &d->cnt, &d->off, &d->xs, &d->key, &d->rank,
                 &d->bcount, &d->boff, &d->order, &d->df, &d->cov, &d->pre, &d->gcov, &d->scan_tmp,
                 &d->gfix};
    for (Buf *b : bs)
        if (b->p) (void)hipFree(b->p);
    if (d->done_ev) (void)hipEventDestroy(d->done_ev);
    delete d;
    return SL_OK;
}

const char *sl_diff_last_error(sl_diff *d) { return d ? d->err.c_str() : "null handle"; }

int sl_diff_forward(sl_diff *d, const float *points, const float *colors, float *image, int keep_for_backward,
                    void *stream) {
    if (!d || !points || !colors || !image) return SL_E_ARG;
    if (hipSetDevice(d->device) != hipSuccess) return dfail(d, SL_E_HIP, "hipSetDevice failed");
    hipStream_t s = (hipStream_t)stream;
    if (int rc0 = diff_order(d, s)) return rc0;
    const DiffDev D = dev_view(d);
    const float2 *pts = (const float2 *)points;
    const uint32_t C = d->C;
    const uint32_t NBK = d->P * (uint32_t)(d->H * d->S);
    const size_t NP = (size_t)d->W * d->H;
    int rc;
    if ((rc = dens(d, d->cnt, ((size_t)C + 1) * 4)) || (rc = dens(d, d->off, ((size_t)C + 1) * 4)) ||
        (rc = dens(d, d->bcount, ((size_t)NBK + 1) * 4)) || (rc = dens(d, d->boff, ((size_t)NBK + 1) * 4)) ||
        (rc = dens(d, d->cov, (size_t)d->P * NP * 4)) ||
        (rc = dens(d, d->scan_tmp, sl::scan_tmp_elems_needed(std::max<size_t>(C, NBK) + 1) * 4)))
        return rc;
    hipLaunchKernelGGL(k_d_count, dim3(nblk(C, 256)), dim3(256), 0, s, D, pts, BP<uint32_t>(d->cnt));
    sl::scan_exclusive_u32(BP<uint32_t>(d->cnt), BP<uint32_t>(d->off), C, BP<uint32_t>(d->scan_tmp), s);
    uint32_t NX = 0;
    if (hipMemcpyAsync(&NX, BP<uint32_t>(d->off) + C, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return dfail(d, SL_E_HIP, "crossing count read-back failed");
    d->NX = NX;
    if ((rc = dens(d, d->xs, (size_t)NX * sizeof(Cross))) || (rc = dens(d, d->key, (size_t)NX * 4)) ||
        (rc = dens(d, d->rank, (size_t)NX * 4)) || (rc = dens(d, d->order, (size_t)NX * 4)) || (rc = dens(d, d->df, NX)))
        return rc;
    sl::launch_fill_u32(BP<uint32_t>(d->bcount), 0u, NBK, s);
    if (NX) {
        hipLaunchKernelGGL(k_d_cross, dim3(nblk(NX, 256)), dim3(256), 0, s, D, pts, (const uint32_t *)BP<uint32_t>(d->off),
                           NX, BP<Cross>(d->xs), BP<uint32_t>(d->key), BP<uint32_t>(d->rank), BP<uint32_t>(d->bcount));
    }
    sl::scan_exclusive_u32(BP<uint32_t>(d->bcount), BP<uint32_t>(d->boff), NBK, BP<uint32_t>(d->scan_tmp), s);
    if (NX) {
        hipLaunchKernelGGL(k_d_scatter, dim3(nblk(NX, 256)), dim3(256), 0, s, NX, (const uint32_t *)BP<uint32_t>(d->key),
                           (const uint32_t *)BP<uint32_t>(d->rank), (const uint32_t *)BP<uint32_t>(d->boff),
                           BP<uint32_t>(d->order));
    }
    hipLaunchKernelGGL(k_d_fill, dim3(nblk((int64_t)d->P * d->H, 4)), dim3(256), 0, s, D,
                       (const uint32_t *)BP<uint32_t>(d->boff), (const uint32_t *)BP<uint32_t>(d->order),
                       (const Cross *)BP<Cross>(d->xs), BP<uint8_t>(d->df), BP<float>(d->cov));
    float4 *pre = nullptr;
    if (keep_for_backward) {
        if ((rc = dens(d, d->pre, (size_t)d->P * NP * 16))) return rc;
        pre = BP<float4>(d->pre);
    }
    hipLaunchKernelGGL(k_d_composite, dim3(nblk((int64_t)NP, 256)), dim3(256), 0, s, D, (const float *)BP<float>(d->cov),
                       (const float4 *)colors, pre, (float4 *)image);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return dfail(d, SL_E_HIP, "forward launch failed: %s", hipGetErrorString(e));
    d->have_pre = keep_for_backward != 0;
    d->last_points = points;
    d->last_colors = colors;
    return diff_issued(d, s);
}

int sl_diff_backward(sl_diff *d, const float *grad_image, float *grad_points, float *grad_colors, void *stream) {
    if (!d || !grad_image || !grad_points || !grad_colors) return SL_E_ARG;
    if (!d->have_pre) return dfail(d, SL_E_STATE, "backward needs a forward with keep_for_backward");
    if (hipSetDevice(d->device) != hipSuccess) return dfail(d, SL_E_HIP, "hipSetDevice failed");
    hipStream_t s = (hipStream_t)stream;
    if (int rc0 = diff_order(d, s)) return rc0;
    const DiffDev D = dev_view(d);
    const size_t NP = (size_t)d->W * d->H;
    int rc;
    const size_t npt = (size_t)d->V * 2, ncol = (size_t)d->P * 4;
    if ((rc = dens(d, d->gcov, (size_t)d->P * NP * 4)) || (rc = dens(d, d->gfix, (npt + ncol) * 8))) return rc;
    unsigned long long *fix_pts = BP<unsigned long long>(d->gfix), *fix_col = fix_pts + npt;
    hipLaunchKernelGGL(k_d_clear, dim3(256), dim3(256), 0, s, BP<float>(d->gfix), (npt + ncol) * 2);
    hipLaunchKernelGGL(k_d_back_pixels, dim3(nblk((int64_t)NP, 256)), dim3(256), 0, s, D, (const float *)BP<float>(d->cov),
                       (const float4 *)d->last_colors, (const float4 *)BP<float4>(d->pre), (const float4 *)grad_image,
                       BP<float>(d->gcov), fix_col);
    if (d->NX) {
        hipLaunchKernelGGL(k_d_back_cross, dim3(d->C, shares_of(d->NX, d->C)), dim3(64), 0, s, D, (const uint32_t *)BP<uint32_t>(d->off),
                           (const Cross *)BP<Cross>(d->xs), (const uint8_t *)BP<uint8_t>(d->df),
                           (const float2 *)d->last_points, (const float *)BP<float>(d->gcov), fix_pts);
    }
    hipLaunchKernelGGL(k_d_unfix, dim3(256), dim3(256), 0, s, (const long long *)fix_pts, grad_points, npt);
    hipLaunchKernelGGL(k_d_unfix, dim3(16), dim3(256), 0, s, (const long long *)fix_col, grad_colors, ncol);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return dfail(d, SL_E_HIP, "backward launch failed: %s", hipGetErrorString(e));
    return diff_issued(d, s);
}

int sl_diff_crossings(sl_diff *d, int64_t *n) {
    if (!d || !n) return SL_E_ARG;
    *n = d->NX;
    return SL_OK;
}

}  // extern "C"
