// sl_resolve.hip -- per-(path, row) resolve: order a bucket's fragments by cell x, run
// the winding scan, merge fragments of a cell into one per-sample stencil mask and
// emit interior spans.  Together these replace the reference's segmented sort
// (cuda_seg_sort_int_by_int), int8 winding scan (thrust_impl_scan.cu:16-19),
// k_mark_merged_fragment_and_span (.cu:462-535), k_gen_stencil_cuda_sm /
// k_gen_stencil_block_boundary (.cu:554-786) and k_gen_gl_merged_fragment_and_span
// (.cu:789-868).
//
// What a bucket leaves for the compositors, at its own stretch of arrays indexed by fragment
// (base = boff[bucket]; it has at most as many merged cells as fragments):
//   icov / imask [base + m]  sample counts / mask of its m-th merged 2x2 cell, in x order;
//   prec [base + e]          per 64-pixel tile holding merged cells, in x order: {cells
//                            covered by a span or merged, merged cells (bit c: the tile's
//                            c-th 2-pixel cell), merged cells before the tile, tile | a span
//                            runs on past the tile << 31 (kept for buckets wider than 63 tiles)};
//   rext, rrec, rtile [place in the row lists]  extent; {colour, records, base, path}; tiles
//                            with a record and tiles wholly inside a span, 64 bits each, bit k
//                            the k-th tile from the extent's first, bit 63 that or any beyond;
//   bcnt [bucket]            {items, merged cells}.
// A column finds its covering item with two bit tests, and a merged cell's index with one
// population count.  For the parity dumps a bucket's items are also listed (one u32 each, x
// of the first pixel | span width << 16, 0 for a merged cell).
#include "sl_device.h"
#include "sl_internal.h"
#include "sl_tables.h"

#include <algorithm>

namespace sl {
using namespace dev;

namespace {

template <int SPP> struct Words { static constexpr int n = SPP == 8 ? 1 : (SPP == 16 ? 2 : 4); };

// fill-rule test of k_mark_merged_fragment_and_span (.cu:511)
__device__ __forceinline__ bool fill_test(int rule, int8_t w) {
    return (rule == 0 && w != 0) || (rule == 1 && (w & 1));
}

// Per-sample stencil of one merged fragment in the reference's 7-bit byte-lane counters:
// acc = init_pos - init_neg + sum(+/- ((mask >> b) & 0x01010101)) (mod 2^32), result bit =
// ((0x80808080 + acc) & 0x7f7f7f7f) tested per byte (k_gen_stencil_cuda_sm, .cu:665-716).
template <int NW>
struct Stencil {
    uint32_t acc[NW][8];
    __device__ __forceinline__ void init(int8_t w) {
        uint32_t ip = 0u, in = 0u;
        if (w < 0) in = 0x01010101u * (uint32_t)(-(int)w);
        else ip = 0x01010101u * (uint32_t)w;
        const uint32_t v = ip - in;
#pragma unroll
        for (int k = 0; k < NW; ++k)
#pragma unroll
            for (int b = 0; b < 8; ++b) acc[k][b] = v;
    }
    __device__ __forceinline__ void add(const uint32_t *m, bool neg) {
#pragma unroll
        for (int k = 0; k < NW; ++k)
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                uint32_t a = (m[k] >> b) & 0x01010101u;
                acc[k][b] = neg ? acc[k][b] - a : acc[k][b] + a;
            }
    }
    // per byte lane: v = (0x80 + counter) & 0x7f; nonzero keeps v != 0, even-odd keeps
    // bit 0.  v <= 0x7f, so v + 0x7f carries into bit 7 of its own byte exactly when v != 0.
    __device__ __forceinline__ void finish(int rule, uint32_t *out) const {
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            uint32_t ret = 0u;
            if (rule == 0) {
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint32_t v = (0x80808080u + acc[k][b]) & 0x7f7f7f7fu;
                    ret |= ((v + 0x7f7f7f7fu) & 0x80808080u) >> (7 - b);
                }
            } else {
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint32_t v = (0x80808080u + acc[k][b]) & 0x7f7f7f7fu;
                    ret |= (v & 0x01010101u) << b;
                }
            }
            out[k] = ret;
        }
    }
};

// The same result for small groups, bit-sliced.  The byte lanes of the stencil word start
// at w * 0x01010101 and gain +/- 0x01 at set bits, so the word is sum_j c_j * 256^j
// (mod 2^32) with c_j the sample's true count w + d_j.  While every c_j lies in
// [-128, 127], adding 0x80808080 leaves byte j = c_j + 128 with no carry between lanes,
// and the tests read c_j mod 128 != 0 (nonzero) or c_j & 1 (even-odd).  With g members and
// |w| <= 127 - g, c_j lies in [-127, 127], so it is enough to count d_j in [-g, g] in P
// two's-complement bit planes, g < 2^(P - 1): nonzero is d_j != -w, even-odd is d_j ^ w in
// plane 0.  Four planes take groups of up to 7, six of up to 31 (crowded rows: a bucket with
// one group of 8 waited for a byte-lane pass over each of its words); larger groups and
// windings take the byte-lane stencil.
__device__ __forceinline__ bool sliced_ok(int g, int8_t w, int planes) {
    const int lim = (1 << (planes - 1)) - 1;
    return g <= lim && w >= lim - 127 && w <= 127 - lim;
}

template <int NW, int P>
struct Sliced {
    uint32_t d[P][NW];
    // d = +1 or -1 (all planes set) at the set bits of one member
    __device__ __forceinline__ void init_one(const uint32_t *m, bool neg) {
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            d[0][k] = m[k];
#pragma unroll
            for (int p = 1; p < P; ++p) d[p][k] = neg ? m[k] : 0u;
        }
    }
    // d += 1 (or -= 1) at the set bits: ripple carry (borrow) through the planes
    __device__ __forceinline__ void add(const uint32_t *m, bool neg) {
        const uint32_t nm = neg ? ~0u : 0u;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            uint32_t c = m[k];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const uint32_t t = (d[p][k] ^ nm) & c;
                d[p][k] ^= c;
                c = t;
            }
        }
    }
    __device__ __forceinline__ void finish(int rule, int8_t w, uint32_t *out) const {
        if (rule != 0) {
            const uint32_t odd = (w & 1) ? ~0u : 0u;
#pragma unroll
            for (int k = 0; k < NW; ++k) out[k] = d[0][k] ^ odd;
            return;
        }
        const int t = -(int)w;
        const bool hit = t >= -(1 << (P - 1)) && t < (1 << (P - 1));  // d_j can equal -w only then
        uint32_t tp[P];
#pragma unroll
        for (int p = 0; p < P; ++p) tp[p] = ((t >> p) & 1) ? ~0u : 0u;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            uint32_t ne = 0u;
#pragma unroll
            for (int p = 0; p < P; ++p) ne |= d[p][k] ^ tp[p];
            out[k] = hit ? ne : ~0u;
        }
    }
};

// Sample counts of the four pixels of a resolved cell mask, 6 bits each at bit 6*(dx*2+dy).
template <int SPP>
__device__ __forceinline__ uint32_t cell_counts(const uint32_t *m) {
    uint32_t c = 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t bits;
        if (SPP == 8) bits = (m[0] >> (q * 8)) & 0xFFu;
        else if (SPP == 16) bits = (m[q >> 1] >> ((q & 1) * 16)) & 0xFFFFu;
        else bits = m[q];
        c |= (uint32_t)__popc(bits) << (6 * q);
    }
    return c;
}

template <int NW>
__device__ __forceinline__ void store_mask(uint32_t *imask, size_t slot, const uint32_t *m) {
    if (NW == 4) *(uint4 *)(imask + slot * 4) = make_uint4(m[0], m[1], m[2], m[3]);
    else if (NW == 2) *(uint2 *)(imask + slot * 2) = make_uint2(m[0], m[1]);
    else imask[slot] = m[0];
}
template <int NW>
__device__ __forceinline__ void load_mask(const uint32_t *p, size_t slot, uint32_t *m) {
    if (NW == 4) { uint4 q = *(const uint4 *)(p + slot * 4); m[0] = q.x; m[1] = q.y; m[2] = q.z; m[3] = q.w; }
    else if (NW == 2) { uint2 q = *(const uint2 *)(p + slot * 2); m[0] = q.x; m[1] = q.y; }
    else m[0] = p[slot];
}

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

struct ResolveArgs {
    int64_t NB;
    const int2 *binfo;
    const uint32_t *boff;
    const uint32_t *bcarry;
    const uint8_t *frule;
    uint32_t *rec;
    int64_t F;
    uint32_t *scratch;
    int W;
    const int4 *pcanvas;     // batched scenes: per-path canvas (W, H, row base, scene)
    const uint32_t *scarry;  // batched scenes: winding-scan carry at each scene's first bucket
    uint32_t *items;         // [2F] item lists, null unless parity dumps are on
    uint32_t *imask;         // written by the KEEP kernels only
    uint32_t *icov;
    uint4 *prec;
    const uint32_t *rpos;    // places in the row lists
    const uint32_t *finfo;   // fill words
    uint32_t *rext;
    uint4 *rrec;
    ulonglong2 *rtile;
    uint2 *bcnt;
    uint32_t *big_list;
    uint32_t *big_count;     // cleared at the frame's start
};

// bits of tiles [t0, t1] counted from tile tb (t0 <= t1), tiles from the 63rd on in bit 63
__device__ __forceinline__ uint64_t tile_bits(int t0, int t1, int tb) {
    return (~0ull << tmin(t0 - tb, 63)) & (~0ull >> (63 - tmin(t1 - tb, 63)));
}
// cells [c0, c1) of a tile, 0 <= c0 < c1 <= 32
__device__ __forceinline__ uint32_t cell_bits(int c0, int c1) { return (~0u << c0) & (~0u >> (32 - c1)); }

constexpr int kBigStage = 16;  // chunks of 64 fragments staged in LDS

// A bucket's results, collected in LDS while it is resolved.
struct BucketOut {
    unsigned long long et, ft;  // tiles with a record, tiles wholly inside a span
    uint32_t ext, nrec, items, merged;
};

__device__ __forceinline__ void out_clear(BucketOut &o) {
    o.et = o.ft = 0ull;
    o.ext = 0xFFFFu;
    o.nrec = o.items = o.merged = 0u;
}

// A bucket's entry in the row lists, by one lane.
__device__ __forceinline__ void put_row(const ResolveArgs &A, int64_t b, uint32_t at, uint32_t base, uint32_t path,
                                        uint32_t colour, const BucketOut &o) {
    A.bcnt[b] = make_uint2(o.items, o.merged);
    if (at == 0xFFFFFFFFu) return;  // the out-of-canvas bucket
    A.rext[at] = o.ext;
    if (!o.items) return;           // an empty extent: the rest is never read
    A.rrec[at] = make_uint4(colour, o.nrec, base, path);
    A.rtile[at] = make_ulonglong2(o.et, o.ft);
}

// What a lane contributes to its bucket's records: its group head's merged cell at x (if any)
// and the span [prev_x + 2, x) before it (if any).  prev_ok: the group before it was merged.
// A record's run of lanes starts at its leader (the first merged cell of its tile); the cells
// of a run are disjoint bits, so their union is a sum, taken from a plain prefix sum.
struct Lane {
    bool merged, span, prev_ok, leader;
    int x, prev_x;
    uint32_t eb;             // its merged cell
    uint32_t co, cp;         // cells it covers in its own run's tile and (leaders) in the run's before
    int f0, f1;              // tiles wholly inside the span: [f0, f1]
    __device__ __forceinline__ void init(bool m, bool s, bool has_prev, int x_, int px, int W) {
        merged = m;
        span = s;
        x = x_;
        prev_x = px;
        prev_ok = has_prev && px >= 0 && px < W;
        leader = merged && !(prev_ok && (px >> 6) == (x >> 6));
        eb = merged ? 1u << ((x & 63) >> 1) : 0u;
        co = eb;
        cp = 0u;
        f0 = 1;
        f1 = 0;
        if (span) {
            const int a = px + 2, ta = a >> 6, tb = (x - 1) >> 6;
            const bool pr = prev_ok && (px >> 6) == ta, ow = merged && (x >> 6) == tb;
            const uint32_t after = pr ? cell_bits((a & 63) >> 1, tmin(x - ta * 64, 64) >> 1) : 0u;
            const uint32_t before = ow && !(pr && ta == tb) ? cell_bits(ta == tb ? (a & 63) >> 1 : 0, (x & 63) >> 1) : 0u;
            co |= before;
            if (leader) cp = after; else co |= after;
            f0 = pr ? ta + 1 : ta;
            f1 = ow ? tb - 1 : tb;
        }
    }
    __device__ __forceinline__ int lo() const { return span ? prev_x + 2 : x; }   // first pixel of its items
    __device__ __forceinline__ int hi() const { return merged ? x + 2 : x; }      // past the last
};

__device__ __forceinline__ int scan_add(int x) { return dpp_scan(x, 0, OpAdd()); }
__device__ __forceinline__ int lane63(int x) { return __builtin_amdgcn_readlane(x, 63); }

template <int NW, int P>
__device__ __forceinline__ void group_sliced(const uint32_t *order, const uint32_t *meta, const uint32_t *msk, int p, int e,
                                             const uint32_t *first, bool neg0, int8_t w_at, int rule, uint32_t *res) {
    Sliced<NW, P> st;
    st.init_one(first, neg0);
    uint32_t iq = order[p + 1 < e ? p + 1 : p];
    for (int q = p + 1; q < e; ++q) {
        uint32_t m[NW];
        load_mask<NW>(msk, iq, m);
        const bool neg = ((meta[iq] >> 24) & 1u) != 0u;
        iq = order[q + 1 < e ? q + 1 : q];  // the next member's index loads beside this one's mask
        st.add(m, neg);
    }
    st.finish(rule, w_at, res);
}

// Merged mask of the cell group at sorted positions [p, e) (records staged in LDS).  The
// first member is the head lane's own record i0 (meta m0): most groups have no other.
template <int NW>
__device__ __forceinline__ void group_mask(const uint32_t *order, const uint32_t *meta, const uint32_t *msk, int p,
                                           int e, uint32_t i0, uint32_t m0, int8_t w_at, int rule, uint32_t *res) {
    uint32_t first[NW];
    load_mask<NW>(msk, i0, first);
    const bool neg0 = ((m0 >> 24) & 1u) != 0u;
    if (sliced_ok(e - p, w_at, 4)) {
        group_sliced<NW, 4>(order, meta, msk, p, e, first, neg0, w_at, rule, res);
    } else if (sliced_ok(e - p, w_at, 6)) {
        group_sliced<NW, 6>(order, meta, msk, p, e, first, neg0, w_at, rule, res);
    } else {
        // rare: one word at a time, for eight counters instead of eight a word
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            Stencil<1> st;
            st.init(w_at);
            st.add(first + k, neg0);
            for (int q = p + 1; q < e; ++q) {
                const uint32_t iq = order[q];
                st.add(msk + iq * NW + k, ((meta[iq] >> 24) & 1u) != 0u);
            }
            st.finish(rule, res + k);
        }
    }
}

// Ranks of the keys `mine` among key[0, n), n a multiple of 4 (keys are distinct; unused places
// hold the largest value).  Four keys a read: a read a key, or a cross-lane operation a key,
// kept the LDS pipe busier than the comparisons.
template <int S>
__device__ __forceinline__ void rank_keys(const uint32_t *key, int n, const uint32_t *mine, int *rk) {
#pragma unroll
    for (int s = 0; s < S; ++s) rk[s] = 0;
#pragma unroll 4
    for (int j = 0; j < n; j += 4) {
        const uint4 k = *(const uint4 *)(key + j);
#pragma unroll
        for (int s = 0; s < S; ++s)
            rk[s] += (k.x < mine[s] ? 1 : 0) + (k.y < mine[s] ? 1 : 0) + (k.z < mine[s] ? 1 : 0) + (k.w < mine[s] ? 1 : 0);
    }
}

// A bucket walked in chunks of 64 sorted records: totals, and the cells of the last record,
// which the next chunk may add to.
struct Chunks {
    int nrec = 0, merged = 0, spans = 0, xmin = INT_MAX, xmax = INT_MIN;
    uint32_t cover = 0u, edge = 0u;
};

template <int SPP, bool KEEP>
__device__ __forceinline__ void chunk_emit(const ResolveArgs &A, uint32_t base, const Lane &L, const uint32_t *res,
                                           BucketOut &O, Chunks &K) {
    constexpr int NW = Words<SPP>::n;
    const int lane = threadIdx.x & 63;
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    const uint64_t mm = __ballot(L.merged), sm = __ballot(L.span), lm = __ballot(L.leader);
    const int mi = K.merged + (int)__popcll(mm & lt), li = (int)__popcll(lm & lt);
    const uint32_t pe = (uint32_t)scan_add((int)L.eb), pc = (uint32_t)scan_add((int)L.co);
    uint4 *rec = A.prec + base;
    // the open record takes the lanes before the first leader; a leader closes it
    const int f = lm ? (int)__builtin_ctzll(lm) : 64;
    if (f > 0) {
        K.edge += (uint32_t)__builtin_amdgcn_readlane((int)pe, f - 1);
        K.cover += (uint32_t)__builtin_amdgcn_readlane((int)pc, f - 1);
    }
    if (lm) {
        K.cover += (uint32_t)__builtin_amdgcn_readlane((int)L.cp, f);
        if (lane == 0 && K.nrec > 0) *(uint2 *)&rec[K.nrec - 1].x = make_uint2(K.cover, K.edge);
        const uint64_t later = lane < 63 ? lm & (~0ull << (lane + 1)) : 0ull;
        const int last = later ? (int)__builtin_ctzll(later) - 1 : 63;
        const uint32_t e = (uint32_t)__shfl((int)pe, last, 64) - (pe - L.eb);
        const uint32_t nc = (uint32_t)__shfl((int)L.cp, (last + 1) & 63, 64);
        const uint32_t c = (uint32_t)__shfl((int)pc, last, 64) - (pc - L.co) + (later ? nc : 0u);
        if (L.leader) rec[K.nrec + li] = make_uint4(c, e, (uint32_t)mi, (uint32_t)(L.x >> 6));
        const int ol = 63 - (int)__builtin_clzll(lm);  // the last leader's record stays open
        K.cover = (uint32_t)__builtin_amdgcn_readlane((int)c, ol);
        K.edge = (uint32_t)__builtin_amdgcn_readlane((int)e, ol);
    }
    if (mm | sm) {
        const int first = (int)__builtin_ctzll(mm | sm), last = 63 - (int)__builtin_clzll(mm | sm);
        K.xmin = tmin(K.xmin, __builtin_amdgcn_readlane(L.lo(), first));
        K.xmax = tmax(K.xmax, __builtin_amdgcn_readlane(L.hi(), last));
        const int tb = K.xmin >> 6;
        if (L.leader) atomicOr(&O.et, 1ull << tmin((L.x >> 6) - tb, 63));
        if (L.f0 <= L.f1) atomicOr(&O.ft, tile_bits(L.f0, L.f1, tb));
    }
    const bool far = L.f0 <= L.f1 && L.prev_ok && L.f1 - (K.xmin >> 6) >= 63;
    if (__ballot(far)) {
        __threadfence();  // the record's tile is stored
        if (far) atomicOr(&rec[K.nrec - 1 + li].w, 0x80000000u);
    }
    if (KEEP && A.items) {
        const size_t it = 2 * (size_t)base + (size_t)(mi + K.spans + (int)__popcll(sm & lt));
        if (L.span) A.items[it] = (uint32_t)(L.prev_x + 2) | ((uint32_t)(L.x - L.prev_x - 2) << 16);
        if (L.merged) A.items[it + (L.span ? 1 : 0)] = (uint32_t)L.x;
    }
    if (L.merged) {
        if (KEEP) store_mask<NW>(A.imask, (size_t)base + mi, res);
        A.icov[base + mi] = cell_counts<SPP>(res);
    }
    K.nrec += (int)__popcll(lm);
    K.merged += (int)__popcll(mm);
    K.spans += (int)__popcll(sm);
}

__device__ __forceinline__ void chunks_end(const ResolveArgs &A, uint32_t base, BucketOut &O, const Chunks &K) {
    if ((threadIdx.x & 63) == 0) {
        if (K.nrec) *(uint2 *)&A.prec[base + K.nrec - 1].x = make_uint2(K.cover, K.edge);
        if (K.merged + K.spans > 0) O.ext = (uint32_t)K.xmin | ((uint32_t)K.xmax << 16);
        O.nrec = (uint32_t)K.nrec;
        O.items = (uint32_t)(K.merged + K.spans);
        O.merged = (uint32_t)K.merged;
    }
    wave_sync_lds();
}

// Resolve one (path, row) bucket of n <= 64*S*WAVES fragments with a block of WAVES waves: stage
// the records in LDS, rank them by (cell x, index), then the first wave walks the sorted order
// in chunks of 64 carrying the winding number and the records (the others return).  Per cell
// group, the first lane sums the members' masks into the per-sample stencil; spans open between
// groups whose winding passes the fill rule.
template <int SPP, int S, bool KEEP, int WAVES = 1>
__device__ __forceinline__ void resolve_bucket(const ResolveArgs &A, int64_t b, uint32_t base, int n, uint32_t *key,
                                               uint32_t *order, uint32_t *meta, uint32_t *msk,
                                               unsigned long long *ghead, BucketOut &O) {
    constexpr int NW = Words<SPP>::n;
    const int lane = threadIdx.x & 63, tid = threadIdx.x;
    constexpr int T = 64 * WAVES;
    uint32_t mykey[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int i = s * T + tid;
        mykey[s] = 0xFFFFFFFFu;
        if (i < n) {
            uint32_t mk[NW];
            const uint32_t m = Records<NW>{A.rec, A.F}.load((size_t)base + i, mk);
            meta[i] = m;
            store_mask<NW>(msk, (size_t)i, mk);
            mykey[s] = ((m & 0xFFFFu) << 10) | (uint32_t)i;
        }
        key[i] = mykey[s];
    }
    __syncthreads();
    int rk[S];
    rank_keys<S>(key, (n + 3) & ~3, mykey, rk);
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s * T + tid < n) order[rk[s]] = (uint32_t)(s * T + tid);
    __syncthreads();
    // group heads of every chunk as wave masks: a group ends at the next head
    const int nc = (n + 63) >> 6;
#pragma unroll 1
    for (int c = tid >> 6; c < nc; c += WAVES) {
        const int p = c * 64 + lane;
        bool h = false;
        if (p < n) h = p == 0 || (meta[order[p]] & 0xFFFFu) != (meta[order[p - 1]] & 0xFFFFu);
        const uint64_t hm = __ballot(h);
        if (lane == 0) ghead[c] = hm;
    }
    __syncthreads();
    if (WAVES > 1 && tid >= 64) return;

    const int rule = A.frule[A.binfo[b].x];
    uint32_t wcarry = A.bcarry[b];
    int W = A.W;
    if (A.pcanvas) {
        // each scene of a batch scans its winding numbers from zero
        const int4 cv = A.pcanvas[A.binfo[b].x];
        W = cv.x;
        wcarry -= A.scarry[cv.w];
    }
    Chunks K;
#pragma unroll 1
    for (int c = 0; c < nc; ++c) {
        const int p = c * 64 + lane;
        const bool v = p < n;
        const uint32_t i = v ? order[p] : 0u;
        const uint32_t m = v ? meta[i] : 0u;
        const int cx = (int)(m & 0xFFFFu);
        const int swn = v ? (int)(int8_t)(m >> 16) : 0;
        const int prev_cx = (v && p > 0) ? (int)(meta[order[p - 1]] & 0xFFFFu) : -1;
        const bool head = v && (p == 0 || cx != prev_cx);
        const int incl = scan_add(swn);
        const int8_t w_at = (int8_t)(int)(wcarry + (uint32_t)(incl - swn));
        wcarry += (uint32_t)lane63(incl);
        const int x = 2 * cx - 2;
        const bool merged = head && x >= 0 && x < W;
        uint32_t res[NW];
        if (merged) {
            const uint64_t later = lane < 63 ? (ghead[c] & (~0ull << (lane + 1))) : 0ull;
            int e = n;
            if (later) {
                e = c * 64 + (int)__builtin_ctzll(later);
            } else {
                for (int c2 = c + 1; c2 < nc; ++c2)
                    if (ghead[c2]) { e = c2 * 64 + (int)__builtin_ctzll(ghead[c2]); break; }
            }
            group_mask<NW>(order, meta, msk, p, e, i, m, w_at, rule, res);
        }
        const int prev_x = 2 * prev_cx - 2;
        Lane L;
        L.init(merged, head && p > 0 && (prev_x + 2 < x) && fill_test(rule, w_at), p > 0, x, prev_x, W);
        chunk_emit<SPP, KEEP>(A, base, L, res, O, K);
    }
    chunks_end(A, base, O, K);
}

constexpr int64_t kResolveWaves = 10240;  // at least this many waves (see launch_resolve)

// A wave-wide ballot as seen by a lane of a segment of S lanes: its segment's bits, bit i the
// segment's i-th lane.  Packed segments lie in one half of the ballot, so 32 bits do.
template <int S> struct SegBits {
    uint64_t m;
    __device__ __forceinline__ SegBits(bool v) : m(__ballot(v)) {}
    __device__ __forceinline__ int below(int i) const { return (int)__popcll(m & (i ? (~0ull >> (64 - i)) : 0ull)); }
    __device__ __forceinline__ int count() const { return (int)__popcll(m); }
    __device__ __forceinline__ int first() const { return (int)__builtin_ctzll(m); }
    __device__ __forceinline__ int last() const { return 63 - (int)__builtin_clzll(m); }
    // the first set bit after i, or S
    __device__ __forceinline__ int after(int i) const {
        const uint64_t l = i < 63 ? m & (~0ull << (i + 1)) : 0ull;
        return l ? (int)__builtin_ctzll(l) : S;
    }
};
template <int S> struct SegBits32 {
    uint32_t m;
    __device__ __forceinline__ SegBits32(bool v) {
        const uint64_t b = __ballot(v);
        const int lane = threadIdx.x & 63;
        m = lane & 32 ? (uint32_t)(b >> 32) : (uint32_t)b;
        if (S == 16) m = (m >> (lane & 16)) & 0xFFFFu;
    }
    __device__ __forceinline__ int below(int i) const { return __popc(m & ((1u << i) - 1u)); }
    __device__ __forceinline__ int count() const { return __popc(m); }
    __device__ __forceinline__ int first() const { return __ffs((int)m) - 1; }
    __device__ __forceinline__ int last() const { return 31 - __clz((int)m); }
    __device__ __forceinline__ int after(int i) const {
        const uint32_t l = m & ~((2u << i) - 1u);  // i = 31: no bits
        return l ? __ffs((int)l) - 1 : S;
    }
};
template <> struct SegBits<32> : SegBits32<32> { using SegBits32<32>::SegBits32; };
template <> struct SegBits<16> : SegBits32<16> { using SegBits32<16>::SegBits32; };

// The records of the buckets in a wave's 64 / S segments, each bucket in one pass.
template <int SPP, int S, bool KEEP>
__device__ __forceinline__ void segment_emit(const ResolveArgs &A, bool live, uint32_t base, const Lane &L,
                                             const uint32_t *res, BucketOut &O) {
    constexpr int NW = Words<SPP>::n;
    const int lane = threadIdx.x & 63;
    const int i = lane % S, seg = lane / S, sb = seg * S;
    const SegBits<S> mm(L.merged), sm(L.span), lm(L.leader), any(L.merged || L.span);
    const int mi = mm.below(i), li = lm.below(i);
    if (L.merged) {
        if (KEEP) store_mask<NW>(A.imask, (size_t)base + mi, res);
        A.icov[base + mi] = cell_counts<SPP>(res);
    }
    // extent: the first and the last lane with an item
    int xmin, xmax;
    if (S == 64) {
        xmin = __builtin_amdgcn_readlane(L.lo(), any.m ? any.first() : 0);
        xmax = __builtin_amdgcn_readlane(L.hi(), any.m ? any.last() : 0);
    } else {
        xmin = __shfl(L.lo(), any.m ? sb + any.first() : lane, 64);
        xmax = __shfl(L.hi(), any.m ? sb + any.last() : lane, 64);
    }
    const int tb = xmin >> 6;
    if (L.leader) atomicOr(&O.et, 1ull << tmin((L.x >> 6) - tb, 63));
    if (L.f0 <= L.f1) atomicOr(&O.ft, tile_bits(L.f0, L.f1, tb));
    // a leader's record: the sums of its run of lanes, up to the next leader
    const uint32_t pe = (uint32_t)dpp_scan_seg<S>((int)L.eb, 0, OpAdd()), pc = (uint32_t)dpp_scan_seg<S>((int)L.co, 0, OpAdd());
    const int next = lm.after(i);
    const uint32_t e = (uint32_t)__shfl((int)pe, sb + next - 1, 64) - (pe - L.eb);
    const uint32_t nc = (uint32_t)__shfl((int)L.cp, (sb + next) & 63, 64);
    const uint32_t c = (uint32_t)__shfl((int)pc, sb + next - 1, 64) - (pc - L.co) + (next < S ? nc : 0u);
    uint4 *rec = A.prec + base;
    if (L.leader) rec[li] = make_uint4(c, e, (uint32_t)mi, (uint32_t)(L.x >> 6));
    const bool far = L.f0 <= L.f1 && L.prev_ok && L.f1 - tb >= 63;
    if (__ballot(far)) {
        __threadfence();  // the record's tile is stored
        if (far) atomicOr(&rec[li - 1].w, 0x80000000u);
    }
    if (KEEP && A.items) {
        const size_t it = 2 * (size_t)base + (size_t)(mi + sm.below(i));
        if (L.span) A.items[it] = (uint32_t)(L.prev_x + 2) | ((uint32_t)(L.x - L.prev_x - 2) << 16);
        if (L.merged) A.items[it + (L.span ? 1 : 0)] = (uint32_t)L.x;
    }
    if (live && i == 0) {
        if (any.m) O.ext = (uint32_t)xmin | ((uint32_t)xmax << 16);
        O.nrec = (uint32_t)lm.count();
        O.items = (uint32_t)(mm.count() + sm.count());
        O.merged = (uint32_t)mm.count();
    }
    __syncthreads();
}

// One small bucket's records, loaded a bucket ahead of its resolve (the grid-stride loop
// keeps the next bucket's records in flight while the current one resolves); the bucket
// scalars come from per-lane registers (see k_resolve_first).
template <int NW>
struct SmallIn {
    uint32_t meta, mk[NW];
    uint32_t carry;
    int rule, W;
};

template <int NW>
__device__ __forceinline__ void small_load(const ResolveArgs &A, uint32_t base, uint32_t end, SmallIn<NW> &o) {
    const int lane = threadIdx.x & 63;
    const int n = (int)(end - base);
    o.meta = 0u;
#pragma unroll
    for (int k = 0; k < NW; ++k) o.mk[k] = 0u;
    if (n > 0 && n <= 64 && lane < n) {
        o.meta = Records<NW>{A.rec, A.F}.load((size_t)base + lane, o.mk);
    }
}

// resolve_bucket<SPP, 1> with the records already in registers
template <int SPP, bool KEEP>
__device__ __forceinline__ void resolve_small(const ResolveArgs &A, uint32_t base, int n,
                                              const SmallIn<Words<SPP>::n> &in, uint32_t *key, uint32_t *order, uint32_t *meta,
                                              uint32_t *msk, BucketOut &O) {
    constexpr int NW = Words<SPP>::n;
    const int lane = threadIdx.x & 63;
    uint32_t mykey = 0xFFFFFFFFu;
    if (lane < n) {
        meta[lane] = in.meta;
        store_mask<NW>(msk, (size_t)lane, in.mk);
        mykey = ((in.meta & 0xFFFFu) << 10) | (uint32_t)lane;
    }
    key[lane] = mykey;
    __syncthreads();
    int rk;
    rank_keys<1>(key, (n + 3) & ~3, &mykey, &rk);
    if (lane < n) order[rk] = (uint32_t)lane;
    __syncthreads();

    const int rule = in.rule;
    uint32_t wcarry = in.carry;
    const int W = in.W;
    const int p = lane;
    const bool v = p < n;
    const uint32_t i = v ? order[p] : 0u;
    const uint32_t m = v ? meta[i] : 0u;
    const int cx = (int)(m & 0xFFFFu);
    const int swn = v ? (int)(int8_t)(m >> 16) : 0;
    const int prev_cx = (v && p > 0) ? (int)(meta[order[p - 1]] & 0xFFFFu) : -1;
    const bool head = v && (p == 0 || cx != prev_cx);
    const int incl = scan_add(swn);
    const int8_t w_at = (int8_t)(int)(wcarry + (uint32_t)(incl - swn));
    const int x = 2 * cx - 2;
    const bool merged = head && x >= 0 && x < W;
    // the group of a head lane ends at the next head (or the bucket end)
    const SegBits<64> heads(head);
    uint32_t res[NW];
    if (merged) group_mask<NW>(order, meta, msk, p, tmin(heads.after(p), n), i, m, w_at, rule, res);
    const int prev_x = 2 * prev_cx - 2;
    Lane L;
    L.init(merged, head && p > 0 && (prev_x + 2 < x) && fill_test(rule, w_at), p > 0, x, prev_x, W);
    segment_emit<SPP, 64, KEEP>(A, true, base, L, res, O);
}

// Buckets of at most S (16 or 32) fragments, 64 / S of them in one wave: lane l works on
// segment l / S, whose records, rank sort, scans and reductions stay inside its S lanes
// (segmented DPP scans), so one pass resolves the whole pack.  ks[s] is the s-th bucket's
// slot in the per-lane scalars (lane k holds bucket b0 + k G), -1 for an empty segment.
template <int SPP, int S, bool KEEP>
__device__ __forceinline__ void resolve_pack(const ResolveArgs &A, const int *ks, int vbase, int vend, int vcarry,
                                             int vrule, int vW, uint32_t *key, uint32_t *order, uint32_t *meta, uint32_t *msk,
                                             BucketOut *out) {
    constexpr int NW = Words<SPP>::n;
    constexpr int P = 64 / S;
    const int lane = threadIdx.x & 63;
    const int seg = lane / S, i = lane % S, sb = seg * S;
    int k = -1;
#pragma unroll
    for (int s = 0; s < P; ++s)
        if (seg == s) k = ks[s];
    // every lane takes part in the cross-lane reads (a lane outside the exec mask would
    // supply zeros to the lanes reading from it)
    const int src = k < 0 ? 0 : k;
    const uint32_t base = (uint32_t)__shfl(vbase, src, 64);
    const int end = __shfl(vend, src, 64);
    const uint32_t wcarry = (uint32_t)__shfl(vcarry, src, 64);
    const int rule = __shfl(vrule, src, 64);
    const int W = __shfl(vW, src, 64);
    const int n = k < 0 ? 0 : end - (int)base;
    uint32_t mykey = 0xFFFFFFFFu;
    if (i < n) {
        uint32_t mk[NW];
        const uint32_t m = Records<NW>{A.rec, A.F}.load((size_t)base + i, mk);
        meta[lane] = m;
        store_mask<NW>(msk, (size_t)lane, mk);
        mykey = ((m & 0xFFFFu) << 10) | (uint32_t)i;
    }
    key[lane] = mykey;
    __syncthreads();
    int rk;
    rank_keys<1>(key + sb, S, &mykey, &rk);
    if (i < n) order[sb + rk] = (uint32_t)lane;  // LDS index of the record
    __syncthreads();

    const int p = i;
    const bool v = p < n;
    const uint32_t i0 = v ? order[sb + p] : 0u;
    const uint32_t m = v ? meta[i0] : 0u;
    const int cx = (int)(m & 0xFFFFu);
    const int swn = v ? (int)(int8_t)(m >> 16) : 0;
    const int prev_cx = (v && p > 0) ? (int)(meta[order[sb + p - 1]] & 0xFFFFu) : -1;
    const bool head = v && (p == 0 || cx != prev_cx);
    const int incl = dpp_scan_seg<S>(swn, 0, OpAdd());
    const int8_t w_at = (int8_t)(int)(wcarry + (uint32_t)(incl - swn));
    const int x = 2 * cx - 2;
    const bool merged = head && x >= 0 && x < W;
    // the group of a head lane ends at the next head of its segment (or the bucket end)
    const SegBits<S> heads(head);
    uint32_t res[NW];
    if (merged) group_mask<NW>(order + sb, meta, msk, p, tmin(heads.after(i), n), i0, m, w_at, rule, res);
    const int prev_x = 2 * prev_cx - 2;
    Lane L;
    L.init(merged, head && p > 0 && (prev_x + 2 < x) && fill_test(rule, w_at), p > 0, x, prev_x, W);
    segment_emit<SPP, S, KEEP>(A, k >= 0, base, L, res, out[src]);
}

// Every bucket: empty ones are cleared, buckets of at most 128 fragments are resolved,
// larger ones are listed for the size-class passes below.  Five waves per SIMD: the records'
// arithmetic spills at six.  On the 2048x2048 illustration (1.8 M buckets) 1.30 ms; writing each
// bucket's results as it ends, 1.57, ranking by cross-lane reads, 1.37, one pack's records
// loaded ahead of their turn, 1.52.
template <int SPP, bool KEEP>
__global__ void __launch_bounds__(64, 5) k_resolve_first(ResolveArgs A) {
    constexpr int NW = Words<SPP>::n;
    __shared__ __align__(16) uint32_t key[128], msk[128 * NW];
    __shared__ uint32_t order[128], meta[128];
    __shared__ unsigned long long ghead[2];
    // results of the wave's 64 buckets, written together at the end: 64 lanes wait for their
    // buckets' places and colours at once, where a lane a bucket would wait at each
    __shared__ BucketOut out[64];
    const int lane = threadIdx.x;
    const int64_t G = gridDim.x;
    // Strided buckets keep the waves' loads balanced (a path's neighbouring rows have
    // similar sizes); the blocks of one XCD take consecutive b0, so neighbouring buckets,
    // whose records share cache lines, are resolved under one L2.
    for (int64_t b0 = xcd_chunk(blockIdx.x, (uint32_t)G); b0 < A.NB; b0 += 64 * G) {
        // The wave's next 64 buckets b0 + k G: lane k loads their offsets and scalars with
        // vector loads, read back per bucket by readlane.  (Scalar loads would share the
        // LDS wait counter, so every LDS wait of a resolve would also wait for them.)
        const int64_t bl = b0 + (int64_t)lane * G;
        int vbase = 0, vend = 0, vcarry = 0, vrule = 0, vW = A.W;
        if (bl < A.NB) {
            const int2 info = A.binfo[bl];
            vbase = (int)A.boff[bl];
            // the out-of-canvas bucket holds records only for the winding carry
            vend = info.y < 0 ? vbase : (int)A.boff[bl + 1];
            vrule = A.frule[info.x];
            uint32_t carry = A.bcarry[bl];
            if (A.pcanvas) {
                const int4 cv = A.pcanvas[info.x];
                vW = cv.x;
                carry -= A.scarry[cv.w];
            }
            vcarry = (int)carry;
        }
        const int64_t left = (A.NB - b0 + G - 1) / G;
        const int nk = (int)(left < 64 ? left : 64);
        // buckets of up to 16 fragments four to a wave, of 17..32 two to a wave
        const int myn = lane < nk ? vend - vbase : -1;
        out_clear(out[lane]);
        __syncthreads();
        if (myn > 128) A.big_list[atomicAdd(A.big_count, 1u)] = (uint32_t)bl;
        uint64_t m16 = __ballot(myn > 0 && myn <= 16);
        uint64_t m32 = __ballot(myn > 16 && myn <= 32);
        uint64_t rest = __ballot(myn > 32 && myn <= 128);
        while (m16) {
            int ks[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                ks[s] = m16 ? (int)__builtin_ctzll(m16) : -1;
                m16 &= m16 - 1ull;
            }
            resolve_pack<SPP, 16, KEEP>(A, ks, vbase, vend, vcarry, vrule, vW, key, order, meta, msk, out);
        }
        while (m32) {
            int ks[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                ks[s] = m32 ? (int)__builtin_ctzll(m32) : -1;
                m32 &= m32 - 1ull;
            }
            resolve_pack<SPP, 32, KEEP>(A, ks, vbase, vend, vcarry, vrule, vW, key, order, meta, msk, out);
        }
        // the rest one by one, the next bucket's records loading during the current one
        SmallIn<NW> in0, in1;
        if (rest) {
            const int k0 = (int)__builtin_ctzll(rest);
            small_load<NW>(A, (uint32_t)__builtin_amdgcn_readlane(vbase, k0),
                           (uint32_t)__builtin_amdgcn_readlane(vend, k0), in0);
        }
        while (rest) {
            const int k = (int)__builtin_ctzll(rest);
            rest &= rest - 1ull;
            const int64_t b = b0 + (int64_t)k * G;
            const uint32_t base = (uint32_t)__builtin_amdgcn_readlane(vbase, k);
            const int n = __builtin_amdgcn_readlane(vend, k) - (int)base;
            if (rest) {
                const int kn = (int)__builtin_ctzll(rest);
                small_load<NW>(A, (uint32_t)__builtin_amdgcn_readlane(vbase, kn),
                               (uint32_t)__builtin_amdgcn_readlane(vend, kn), in1);
            }
            if (n > 64) {
                resolve_bucket<SPP, 2, KEEP>(A, b, base, n, key, order, meta, msk, ghead, out[k]);
            } else {
                in0.carry = (uint32_t)__builtin_amdgcn_readlane(vcarry, k);
                in0.rule = __builtin_amdgcn_readlane(vrule, k);
                in0.W = __builtin_amdgcn_readlane(vW, k);
                resolve_small<SPP, KEEP>(A, base, n, in0, key, order, meta, msk, out[k]);
            }
            in0 = in1;
        }
        if (myn >= 0 && myn <= 128) {
            const uint32_t path = (uint32_t)A.binfo[bl].x;
            put_row(A, bl, A.rpos[bl], (uint32_t)vbase, path, A.finfo[path], out[lane]);
        }
        __syncthreads();
    }
}

// Waves of a block that resolves one listed bucket: they share the ranking, which compares every
// record with every other (1024 batched scenes: 96 us a sample count, by a lone wave 121).
constexpr int kBigWaves = 4, kBigThreads = 64 * kBigWaves;

// Buckets of more than 1024 fragments (rare): bitonic-sort 64-bit (cell x, index) keys,
// held in the bucket's stretch of the record array (4n words; the padded power of two is at
// most 2n), copy the sorted indices into the scratch (the records are written next), then the
// first wave walks the sorted order in chunks of 64 reading the fragments from global memory.
// Any bucket size works.
template <int SPP, bool KEEP>
__global__ void __launch_bounds__(kBigThreads) k_resolve_huge(ResolveArgs A) {
    constexpr int NW = Words<SPP>::n;
    __shared__ BucketOut O;
    const int lane = threadIdx.x & 63, tid = threadIdx.x;
    const uint32_t nbig = *A.big_count;
    for (uint32_t bi = blockIdx.x; bi < nbig; bi += gridDim.x) {
        const int64_t b = A.big_list[bi];
        const uint32_t base = A.boff[b];
        const int n = (int)(A.boff[b + 1] - base);
        if (n <= 64 * kBigStage) continue;
        const Records<NW> recs{A.rec, A.F};
        if (tid == 0) out_clear(O);
        int P2 = 1;
        while (P2 < n) P2 <<= 1;
        uint32_t *khi = (uint32_t *)(A.prec + base);
        uint32_t *klo = khi + P2;
        for (int i = tid; i < P2; i += kBigThreads) {
            khi[i] = (i < n) ? (recs.meta((size_t)base + i) & 0xFFFFu) : 0xFFFFFFFFu;
            klo[i] = (i < n) ? (uint32_t)i : 0xFFFFFFFFu;
        }
        __syncthreads();
        for (int k = 2; k <= P2; k <<= 1) {
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = tid; i < P2; i += kBigThreads) {
                    const int l = i ^ j;
                    if (l > i) {
                        const uint32_t ah = khi[i], al = klo[i], ch = khi[l], cl = klo[l];
                        const bool gt = ah > ch || (ah == ch && al > cl);
                        const bool up = (i & k) == 0;
                        if (gt == up) {
                            khi[i] = ch; klo[i] = cl;
                            khi[l] = ah; klo[l] = al;
                        }
                    }
                }
                __syncthreads();
            }
        }
        uint32_t *order = A.scratch + base;
        for (int i = tid; i < n; i += kBigThreads) order[i] = klo[i];
        __syncthreads();
        if (tid < 64) {
            // sorted fragment indices; a fragment's cell x is in its record
            auto cell_x = [&](int q) { return (int)(recs.meta((size_t)base + order[q]) & 0xFFFFu); };
            const int rule = A.frule[A.binfo[b].x];
            uint32_t wcarry = A.bcarry[b];
            int W = A.W;
            if (A.pcanvas) {
                const int4 cv = A.pcanvas[A.binfo[b].x];
                W = cv.x;
                wcarry -= A.scarry[cv.w];
            }
            Chunks K;
            for (int c0 = 0; c0 < n; c0 += 64) {
                const int p = c0 + lane;
                const bool v = p < n;
                const uint32_t meta = v ? recs.meta((size_t)base + order[p]) : 0u;
                const int cx = (int)(meta & 0xFFFFu);
                const int swn = v ? (int)(int8_t)(meta >> 16) : 0;
                const int prev_cx = (v && p > 0) ? cell_x(p - 1) : -1;
                const bool head = v && (p == 0 || cx != prev_cx);
                const int incl = scan_add(swn);
                const int8_t w_at = (int8_t)(int)(wcarry + (uint32_t)(incl - swn));
                wcarry += (uint32_t)lane63(incl);
                const int x = 2 * cx - 2;
                const bool merged = head && x >= 0 && x < W;
                uint32_t res[NW];
                if (merged) {
                    Stencil<NW> st;
                    st.init(w_at);
                    for (int q = p; q < n; ++q) {
                        const uint32_t j = order[q];
                        uint32_t m2[NW];
                        const uint32_t mq = recs.load((size_t)base + j, m2);
                        if ((int)(mq & 0xFFFFu) != cx) break;
                        st.add(m2, ((mq >> 24) & 1u) != 0u);
                    }
                    st.finish(rule, res);
                }
                const int prev_x = 2 * prev_cx - 2;
                Lane L;
                L.init(merged, head && p > 0 && (prev_x + 2 < x) && fill_test(rule, w_at), p > 0, x, prev_x, W);
                chunk_emit<SPP, KEEP>(A, base, L, res, O, K);
            }
            chunks_end(A, base, O, K);
        }
        if (tid == 0) {
            const uint32_t path = (uint32_t)A.binfo[b].x;
            put_row(A, b, A.rpos[b], base, path, A.finfo[path], O);
        }
        __syncthreads();
    }
}

// The listed buckets (more than 128 fragments), one per block, in one launch so that the
// few long ones overlap: up to 1024 fragments staged in LDS, more in k_resolve_huge (a kernel of
// its own: as a call from this one it cost 30 us of such a batch, for 4 us of a launch).
template <int SPP, bool KEEP>
__global__ void __launch_bounds__(kBigThreads) k_resolve_big(ResolveArgs A) {
    constexpr int NW = Words<SPP>::n;
    __shared__ __align__(16) uint32_t key[64 * kBigStage], msk[64 * kBigStage * NW];
    __shared__ uint32_t order[64 * kBigStage], meta[64 * kBigStage];
    __shared__ unsigned long long ghead[kBigStage];
    __shared__ BucketOut out;
    const uint32_t nbig = *A.big_count;
    for (uint32_t bi = blockIdx.x; bi < nbig; bi += gridDim.x) {
        const int64_t b = A.big_list[bi];
        const uint32_t base = A.boff[b];
        const int n = (int)(A.boff[b + 1] - base);
        if (n > 64 * kBigStage) continue;  // k_resolve_huge's
        if (threadIdx.x == 0) out_clear(out);
        __syncthreads();
        if (n <= 256) resolve_bucket<SPP, 1, KEEP, kBigWaves>(A, b, base, n, key, order, meta, msk, ghead, out);
        else if (n <= 512) resolve_bucket<SPP, 2, KEEP, kBigWaves>(A, b, base, n, key, order, meta, msk, ghead, out);
        else resolve_bucket<SPP, 4, KEEP, kBigWaves>(A, b, base, n, key, order, meta, msk, ghead, out);
        if (threadIdx.x == 0) {
            const uint32_t path = (uint32_t)A.binfo[b].x;
            put_row(A, b, A.rpos[b], base, path, A.finfo[path], out);
        }
        __syncthreads();
    }
}

// Winding-scan carry at the first bucket of every scene of a batch.
__global__ void k_scene_carry(int n, const uint32_t *__restrict__ sfirst, const uint32_t *__restrict__ pbase,
                              const uint32_t *__restrict__ bcarry, uint32_t *scarry) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) scarry[i] = bcarry[pbase[sfirst[i]]];
}

// ---------------------------------------------------------------------------------
// gradient paint (output_32.vert.glsl:55-97, output_32.frag.glsl:45-51; the multisample
// shaders differ only in the x offset of the line ends).  The reference evaluates the
// gradient coordinates at the two ends of each item's line, (x0 + off, y + 1/2) and
// (x0 + w + off, y + 1/2) per pixel row, the rasterizer interpolates them linearly to the
// pixel centre (t = (x - x0 + 1/2) / w), and the fragment shader maps them to the ramp
// parameter c = min(|d|^2 / (sqrt(B^2 + |d|^2 f.z) - B), 1), d = g - f, B = d . f, and
// samples the 1024-wide ramp with linear filtering and clamped edges, sRGB-decoding the
// texels when sRGB correction is on.  The same float operations, in the same order, are
// restated in the oracle.
// ---------------------------------------------------------------------------------
__device__ __forceinline__ float2 grad_coord(const GradDev &G, const float4 &w0, const float4 &w1, float sx, float sy) {
    const float *k = G.ctx;
    const float rdx = (k[0] * sx + k[3] * sy) + k[6];
    const float rdy = (k[1] * sx + k[4] * sy) + k[7];
    const float rdz = (k[2] * sx + k[5] * sy) + k[8];
    const float q = k[12] / rdz;
    const float ox = k[9] + q * rdx, oy = k[10] + q * rdy;
    return make_float2((ox * w0.x + oy * w0.y) + w0.z, (ox * w0.w + oy * w1.x) + w1.y);
}

// A fill word without alpha names gradient slot c - 1; it paints when the slot's ramp scale
// is positive (the shaders' gradient branch), and draws nothing otherwise.
__device__ __forceinline__ bool grad_paints(const GradDev &G, uint32_t c) {
    const uint32_t gi = c - 1u;
    return gi < G.nslots && G.table[3 * gi + 1].w > 0.f;
}

__device__ __forceinline__ float4 ramp_texel(const GradDev &G, int i, int j, const float *dc, const float *da) {
    const uint32_t t = G.ramp[(size_t)j * 1024 + i];
    return make_float4(dc[t & 0xFFu], dc[(t >> 8) & 0xFFu], dc[(t >> 16) & 0xFFu], da[t >> 24]);
}

// Paint of gradient word c at pixel (x, yrow) of an item covering columns [x0, x0 + w) of
// the cell row holding yrow.  dc / da decode a texel's colour and alpha codes.
__device__ __forceinline__ float4 grad_color(const GradDev &G, uint32_t c, int x0, int w, int x, int yrow, const float *dc,
                             const float *da) {
    const uint32_t gi = c - 1u;
    const float4 w0 = G.table[3 * gi], w1 = G.table[3 * gi + 1], w2 = G.table[3 * gi + 2];
    const float sy = (float)(yrow & ~1) + ((yrow & 1) ? 1.5f : 0.5f);
    const float2 ga = grad_coord(G, w0, w1, (float)x0 + G.xoff, sy);
    const float2 gb = grad_coord(G, w0, w1, (float)(x0 + w) + G.xoff, sy);
    const float t = ((float)(x - x0) + 0.5f) / (float)w;
    const float omt = 1.f - t;
    const float gx = ga.x * omt + gb.x * t, gy = ga.y * omt + gb.y * t;
    const float dx = gx - w2.x, dy = gy - w2.y;
    const float A = dx * dx + dy * dy, B = dx * w2.x + dy * w2.y;
    const float den = sqrtf(B * B + A * w2.z) - B;
    float cc = A * (den > 1e-6f ? 1.f / den : 0.f);
    cc = cc < 1.f ? cc : 1.f;
    if (G.rows <= 0) return make_float4(0.f, 0.f, 0.f, 1.f);
    const int ri = __float_as_int(w1.z);
    const float u = ((float)(ri & 1023) + 0.5f) * (1.f / 1024.f) + cc * w1.w;
    const float v = ((float)(ri >> 10) + 0.5f) * G.irh;
    const float tu = u * 1024.f - 0.5f, tv = v * (float)G.rows - 0.5f;
    const float fu = floorf(tu), fv = floorf(tv);
    const float au = tu - fu, av = tv - fv, bu = 1.f - au, bv = 1.f - av;
    const int iu = (int)fu, jv = (int)fv;
    const int i0 = tmin(tmax(iu, 0), 1023), i1 = tmin(tmax(iu + 1, 0), 1023);
    const int j0 = tmin(tmax(jv, 0), G.rows - 1), j1 = tmin(tmax(jv + 1, 0), G.rows - 1);
    const float4 t00 = ramp_texel(G, i0, j0, dc, da), t10 = ramp_texel(G, i1, j0, dc, da);
    const float4 t01 = ramp_texel(G, i0, j1, dc, da), t11 = ramp_texel(G, i1, j1, dc, da);
    float4 o;
    o.x = (t00.x * bu + t10.x * au) * bv + (t01.x * bu + t11.x * au) * av;
    o.y = (t00.y * bu + t10.y * au) * bv + (t01.y * bu + t11.y * au) * av;
    o.z = (t00.z * bu + t10.z * au) * bv + (t01.z * bu + t11.z * au) * av;
    o.w = (t00.w * bu + t10.w * au) * bv + (t01.w * bu + t11.w * au) * av;
    return o;
}

// ---------------------------------------------------------------------------------
// coverage-mode compositor.  The framebuffer state of each pixel is carried as the four
// decoded floats of its 8-bit codes; every blend re-quantises to a code and decodes it
// again, exactly as an 8-bit framebuffer does:
//   UNORM8: code = largest k with v >= (k - 0.5) / 255, i.e. with 510 v - (2k - 1) >= 0 --
//           one fma gives that sign exactly, applied to an estimate that is never too
//           small; decode = RN(k / 255) by a corrected product.
//   sRGB8:  the top bits of v + 2^-5 name one of 645 intervals that grow with v like the
//           thresholds' distances; none holds two thresholds, so the code is the interval's
//           first or the next, and one 16-byte entry {thr, dec, dec_next, code} decides and
//           decodes.  (4096 equal intervals naming a step took a second, dependent LDS read:
//           headline composite 2.20 ms for 2.01, a 1024x768 gradient scene's 0.43 for 0.32.)
// ---------------------------------------------------------------------------------
// v clamped to [0, 1], NaN to 0
__device__ __forceinline__ float unit(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, 1.f); }

// The code is m = floor(255 v + 0.5).  The estimate floor(RN(255 v + 0.5)) is m or m + 1:
// rounding is monotone and the integers m, m + 1 are floats, so RN never crosses below m.
// One exact sign test, RN(510 v + 1 - 2k) < 0 iff v < thr[k], takes the extra one back.
__device__ __forceinline__ float unorm_codef(float v) {
    const float u = unit(v);
    const float k = floorf(__builtin_fmaf(u, 255.f, 0.5f));
    return __builtin_fmaf(u, 510.f, __builtin_fmaf(k, -2.f, 1.f)) < 0.f ? k - 1.f : k;  // u < thr[k]
}
__device__ __forceinline__ int unorm_code(float v) { return (int)unorm_codef(v); }

__device__ __forceinline__ float unorm_decf(float fk) {
    const float r = 1.f / 255.f;
    const float q = fk * r;
    return __builtin_fmaf(__builtin_fmaf(-q, 255.f, fk), r, q);
}
__device__ __forceinline__ float unorm_dec(int k) { return unorm_decf((float)k); }

// the step entry of v's interval (v below 0 or NaN takes the first, above 1 the last)
__device__ __forceinline__ float4 srgb_step(const float4 *step, float v) {
    const float u = __builtin_amdgcn_fmed3f(v + kQuantShift, kQuantShift, 1.f + kQuantShift);
    return step[(__float_as_uint(u) >> 16) - kQuantBase];
}
__device__ __forceinline__ float srgb_dec(const float4 *step, float v) {
    const float4 st = srgb_step(step, v);
    return v >= st.x ? st.z : st.y;
}
__device__ __forceinline__ int srgb_code(const float4 *step, float v, float &dec) {
    const float4 st = srgb_step(step, v);
    const bool up = v >= st.x;
    dec = up ? st.z : st.y;
    return (int)__float_as_uint(st.w) + (up ? 1 : 0);
}

template <bool SRGB>
__device__ __forceinline__ void blend_dec(const float4 *step, float *d, const float4 &src, float a) {
    const float oma = 1.f - a;
    const float v0 = src.x * a + d[0] * oma;
    const float v1 = src.y * a + d[1] * oma;
    const float v2 = src.z * a + d[2] * oma;
    const float va = a * a + d[3] * oma;
    if (SRGB) {
        d[0] = srgb_dec(step, v0);
        d[1] = srgb_dec(step, v1);
        d[2] = srgb_dec(step, v2);
    } else {
        d[0] = unorm_decf(unorm_codef(v0));
        d[1] = unorm_decf(unorm_codef(v1));
        d[2] = unorm_decf(unorm_codef(v2));
    }
    d[3] = unorm_decf(unorm_codef(va));
}

template <bool SRGB>
__device__ __forceinline__ uint32_t pack_dec(const float4 *step, const float *d) {
    uint32_t o = 0u;
    float t;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) o |= (uint32_t)(SRGB ? srgb_code(step, d[ch], t) : unorm_code(d[ch])) << (8 * ch);
    return o | ((uint32_t)unorm_code(d[3]) << 24);
}

struct CovArgs {
    int W, H, tiles_x;
    const uint32_t *rowstart;
    const uint32_t *rext;       // per row-list entry: extent
    const uint4 *rrec;          //   colour, records, base, path
    const ulonglong2 *rtile;    //   tiles with a record, tiles inside a span
    const uint4 *prec;          // records
    const uint32_t *icov;       // sample counts of merged cells
    const uint32_t *imask;      // masks of merged cells (multisample output)
    const uint32_t *ptab;       // per-path blend tables (multisample output)
    const float *dec_c;         // [256] colour decode, for the paint colours
    const float *dec_a;         // [256] alpha decode (gradient ramp texels)
    const float4 *step_c;       // [kQuantSteps] sRGB steps {thr, dec, dec_next, code}
    uint8_t *image;
    int pitch;
    GradDev G;
    // batched scenes: per scene {W, H, first tile, first cell row} and image byte offset
    int nscenes;
    int64_t ntiles;
    const int4 *stile;
    const uint64_t *simg;
};

constexpr int kCovList = 64;    // per-wave list of the tile's buckets

// A bucket's cells in one tile: those covered by a span or merged, the merged ones, and the
// array index of the tile's first merged cell.
struct TileCells {
    uint32_t cover, edge, at;
    int rec;                    // records before the tile; its own is `rec` where has_rec
    bool has_rec;
};

// Whether the row-list entry's bucket has items in the 64-pixel tile `tile` (entry extents
// overlap it), and where its record is.  Tiles from the 63rd of the bucket on are looked up
// in the records themselves.
__device__ __forceinline__ bool tile_hit(const uint4 *__restrict__ prec, uint32_t ext, const uint4 &rec,
                                         const ulonglong2 &bits, int tile, TileCells &t) {
    const int k = tile - (int)((ext & 0xFFFFu) >> 6);
    t.cover = 0xFFFFFFFFu;
    t.edge = 0u;
    t.at = 0u;
    if (k < 63) {
        t.has_rec = (bits.x >> k) & 1ull;
        t.rec = (int)__popcll(bits.x & ((1ull << k) - 1ull));
        return t.has_rec || ((bits.y >> k) & 1ull);
    }
    t.has_rec = false;
    t.rec = 0;
    if (!((bits.x | bits.y) >> 63)) return false;
    int lo = 0, hi = (int)rec.y;  // records of tiles up to this one
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)(prec[rec.z + mid].w & 0x7FFFFFFFu) <= tile) lo = mid + 1; else hi = mid;
    }
    t.rec = lo;
    if (lo == 0) return true;  // before the first merged cell: the span from the canvas edge
    const uint32_t w = prec[rec.z + lo - 1].w;
    if ((int)(w & 0x7FFFFFFFu) != tile) return (w >> 31) != 0u;
    t.has_rec = true;
    t.rec = lo - 1;
    return true;
}

__device__ __forceinline__ void tile_load(const uint4 *__restrict__ prec, uint32_t base, TileCells &t) {
    if (!t.has_rec) return;
    const uint4 r = prec[base + t.rec];
    t.cover = r.x;
    t.edge = r.y;
    t.at = base + r.z;
}

// First pixel and width of the item covering cell c of a tile (gradients run along an item):
// a merged cell, or the span between the merged cells next to it, which may lie in the
// neighbouring records or be missing at the ends of the bucket's extent.  src and ent: the
// bucket's list entries (list_row).
__device__ __forceinline__ void item_extent(const uint4 *__restrict__ prec, const float4 &src, const uint4 &ent, int c,
                                            int tx0, int &x0, int &w) {
    const uint32_t edge = ent.y, prev = __float_as_uint(src.y), next = __float_as_uint(src.z);
    if ((edge >> c) & 1u) {
        x0 = tx0 + 2 * c;
        w = 2;
        return;
    }
    const uint32_t below = edge & ((1u << c) - 1u), above = edge & ~((2u << c) - 1u);
    int end;
    if (below) {
        x0 = tx0 + 2 * (31 - __clz((int)below)) + 2;
    } else if (prev) {
        const uint4 r = prec[prev - 1u];
        x0 = 64 * (int)(r.w & 0x7FFFFFFFu) + 2 * (31 - __clz((int)r.y)) + 2;
    } else {
        x0 = (int)(ent.w & 0xFFFFu);
    }
    if (above) {
        end = tx0 + 2 * (__ffs((int)above) - 1);
    } else if (next) {
        const uint4 r = prec[next - 1u];
        end = 64 * (int)(r.w & 0x7FFFFFFFu) + 2 * (__ffs((int)r.y) - 1);
    } else {
        end = (int)(ent.w >> 16);
    }
    w = end - x0;
}

// Transposes the 32 x 32 bit matrices held by lanes 0-31 and by lanes 32-63: bit c of lane b
// goes to bit b of lane c (c, b within the half).
__device__ __forceinline__ uint32_t transpose32(uint32_t x) {
    const int lane = threadIdx.x & 63;
#define SL_STEP(j, m, fetch)                                                                            \
    {                                                                                                   \
        const uint32_t p = (uint32_t)(fetch);                                                           \
        const bool up = lane & j;                                                                       \
        const uint32_t r = __builtin_amdgcn_alignbit(p, p, up ? j : 32 - j), k = up ? ~(m) : (m);       \
        x = (x & k) | (r & ~k);                                                                         \
    }
#define SL_DPP(c, v) __builtin_amdgcn_update_dpp((int)(v), (int)(v), c, 0xf, 0xf, false)
    SL_STEP(16, 0x0000FFFFu, __builtin_amdgcn_ds_swizzle((int)x, 0x401F))       // lane ^ 16
    SL_STEP(8, 0x00FF00FFu, SL_DPP(0x128, x))                                   // row_ror:8
    SL_STEP(4, 0x0F0F0F0Fu, SL_DPP(0x1B, SL_DPP(0x141, x)))                     // ^ 7, then ^ 3
    SL_STEP(2, 0x33333333u, SL_DPP(0x4E, x))                                    // quad_perm 2,3,0,1
    SL_STEP(1, 0x55555555u, SL_DPP(0xB1, x))                                    // quad_perm 1,0,3,2
#undef SL_DPP
#undef SL_STEP
    return x;
}

// Lists the row's buckets with items in the tile, in path order, and calls flush(n) for every
// full list and the last.  The row's extents are read first, two a lane, and the entries that
// overlap the tile queued; 64 queued entries at a time then load their records.  (Loading
// everything of 64 entries at once took three dependent loads for every 64 buckets of the
// row; on a sheet of glyphs nearly all of them lie beside the tile.)
// A list entry is {paint's colour, alpha * ascale} in l_src and {cover, edge, first merged cell,
// path} in l_ent; a gradient's {its word, the index of the bucket's record before the tile + 1
// (0: none), the same of the next record, -1} and its extent for the path.
constexpr int kRowQueue = 192;

template <bool GRAD, class F>
__device__ __forceinline__ void list_row(const CovArgs &A, uint32_t q0, uint32_t q1, int tx, int tx1, float ascale,
                                         const float *s_dec, uint32_t *queue, float4 *l_src, uint4 *l_ent, const F &flush) {
    const int lane = threadIdx.x & 63, tx0 = tx * 64;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int nlist = 0, nq = 0;
    for (uint32_t qc = q0; qc < q1;) {
        // fill the queue: two entries a lane, in order
        const uint32_t q = qc + 2u * (uint32_t)lane;
        const uint32_t x0 = q < q1 ? A.rext[q] : 0xFFFFu, x1 = q + 1u < q1 ? A.rext[q + 1u] : 0xFFFFu;
        const bool h0 = (int)(x0 & 0xFFFFu) < tx1 && (int)(x0 >> 16) > tx0;
        const bool h1 = (int)(x1 & 0xFFFFu) < tx1 && (int)(x1 >> 16) > tx0;
        const unsigned long long m0 = __ballot(h0), m1 = __ballot(h1);
        const int at = nq + (int)__popcll(m0 & lt) + (int)__popcll(m1 & lt);
        if (h0) queue[at] = q;
        if (h1) queue[at + (h0 ? 1 : 0)] = q + 1u;
        nq += (int)__popcll(m0) + (int)__popcll(m1);
        qc += 128u;
        // and empty it, 64 at a time (all of it at the row's end)
        while (nq >= 64 || (qc >= q1 && nq > 0)) {
            wave_sync_lds();
            const int n = tmin(nq, 64);
            bool ov = false;
            uint4 rec;
            uint32_t ext = 0u;
            TileCells tc;
            if (lane < n) {
                const uint32_t e = queue[lane];
                ext = A.rext[e];
                rec = A.rrec[e];
                // a word without alpha paints nothing, unless it names a gradient that paints
                const bool paints = (rec.x & 0xFF000000u) || (GRAD && rec.x != 0u && grad_paints(A.G, rec.x));
                ov = tile_hit(A.prec, ext, rec, A.rtile[e], tx, tc) && paints;
                if (ov) tile_load(A.prec, rec.z, tc);
            }
            // the queue's remainder moves to its front
            const uint32_t r0 = n + lane < nq ? queue[n + lane] : 0u, r1 = n + 64 + lane < nq ? queue[n + 64 + lane] : 0u;
            wave_sync_lds();
            if (n + lane < nq) queue[lane] = r0;
            if (n + 64 + lane < nq) queue[64 + lane] = r1;
            nq -= n;
            const unsigned long long om = __ballot(ov);
            const int nov = (int)__popcll(om), rank = (int)__popcll(om & lt);
            for (int done = 0; done < nov;) {
                const int take = tmin(kCovList - nlist, nov - done);
                if (ov && rank >= done && rank < done + take) {
                    const int sl = nlist + rank - done;
                    const uint32_t c = rec.x;
                    uint32_t last = rec.w;
                    if (GRAD && !(c & 0xFF000000u)) {
                        const int nx = tc.rec + (tc.has_rec ? 1 : 0);
                        l_src[sl] = make_float4(__uint_as_float(c), __uint_as_float(tc.rec ? rec.z + (uint32_t)tc.rec : 0u),
                                                __uint_as_float(nx < (int)rec.y ? rec.z + (uint32_t)nx + 1u : 0u), -1.f);
                        last = ext;
                    } else {
                        l_src[sl] = make_float4(s_dec[c & 0xFFu], s_dec[(c >> 8) & 0xFFu], s_dec[(c >> 16) & 0xFFu],
                                                unorm_dec((int)(c >> 24)) * ascale);
                    }
                    l_ent[sl] = make_uint4(tc.cover, tc.edge, tc.at, last);
                }
                nlist += take;
                done += take;
                if (nlist == kCovList) {
                    flush(nlist);
                    nlist = 0;
                }
            }
        }
    }
    if (nlist) flush(nlist);
}

// One wavefront per 64x2 pixel tile (lane = pixel column, rows 2r and 2r+1).  The cell
// row's non-empty buckets, in path order, are filtered by extent and tile bitmaps into a
// per-wave list of up to 64 (paint colour decoded, the tile's cells).  The list's cover bits
// are transposed, so that every lane holds the list's buckets covering its column as 64
// bits, and the blend passes run as often as the deepest column's count, each lane taking
// its own next bucket in path order: coverage alpha = paint alpha * covered samples / N
// (output_{8,32}.frag.glsl).  An opaque paint over a whole column leaves its own colour
// exactly, so a column's buckets before its last such one are dropped.
// Bound by the passes' instructions (about 100 each for eight channels; the next pass's
// sample counts load during them).  Seven waves per SIMD (batches six, gradients four): six
// and eight take 1.34 and 1.40 ms for 1.27 on the 2048x2048 illustration.  Finding a column's
// covering item by LDS slots and a max-scan per bucket, in groups of four buckets: 2.01 ms
// there, 543 us for 389 on a 4096x4096 sheet of glyphs, 154 for 23 on a 512x512 drawing of
// opaque cubic chains, 2.5 ms for 0.81 on 1024 such scenes in a batch.
template <int SPP, bool SRGB, bool BATCH, bool GRAD>
__global__ void __launch_bounds__(256, GRAD ? 4 : (BATCH ? 6 : 7)) k_composite_cov(CovArgs A) {
    __shared__ float4 s_step[SRGB ? kQuantSteps : 1];
    __shared__ float s_dec[256];
    __shared__ float s_deca[GRAD ? 256 : 1];
    __shared__ float4 l_src[4][kCovList];
    __shared__ uint4 l_ent[4][kCovList];
    __shared__ uint32_t l_queue[4][kRowQueue];
    for (int i = threadIdx.x; i < 256; i += 256) {
        s_dec[i] = A.dec_c[i];
        if (GRAD) s_deca[i] = A.dec_a[i];
    }
    for (int i = threadIdx.x; i < (SRGB ? kQuantSteps : 0); i += 256) s_step[i] = A.step_c[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int W = A.W, H = A.H, tiles_x = A.tiles_x, row0 = 0, pitch = A.pitch;
    int tile;
    if (!BATCH) {
        // Workgroup b runs on XCD b % 8 (round-robin deal): XCD x takes the cell rows
        // x, x + 8, x + 16, ... whole, its workgroups walking them tile by tile, so each
        // row's records are fetched into one XCD's L2 and every XCD gets rows from the whole
        // image (the per-row work is uneven, so contiguous bands would not balance).
        const int xcd = (int)(blockIdx.x & 7u), t = (int)(blockIdx.x >> 3) * 4 + w;
        const int rr = t / tiles_x, row = xcd + 8 * rr;
        if (row >= (H + 1) / 2) return;
        tile = row * tiles_x + (t - rr * tiles_x);
    } else {
        tile = (int)blockIdx.x * 4 + w;
        if (tile >= A.ntiles) return;
    }
    uint8_t *image = A.image;
    if (BATCH) {
        // the scene whose tile range holds this tile: last one with first tile <= tile
        int lo = 0, hi = A.nscenes - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (A.stile[mid].z <= tile) lo = mid; else hi = mid - 1;
        }
        const int4 st = A.stile[lo];
        W = st.x;
        H = st.y;
        tiles_x = (W + 63) >> 6;
        tile -= st.z;
        row0 = st.w;
        pitch = 4 * W;
        image = A.image + A.simg[lo];
    }
    const int r = tile / tiles_x, tx = tile - r * tiles_x;
    const int tx0 = tx * 64, tx1 = tmin(tx0 + 64, W);
    const int x = tx0 + lane, cell = lane >> 1, half = 12 * (lane & 1);
    constexpr float kInvN = 1.f / (float)SPP;
    constexpr uint32_t kFull = (uint32_t)SPP * 65u;  // both rows' counts
    float d0[4] = {1.f, 1.f, 1.f, 1.f}, d1[4] = {1.f, 1.f, 1.f, 1.f};

    auto flush = [&](int n) {
        wave_sync_lds();
        const uint4 mine = lane < n ? l_ent[w][lane] : make_uint4(0u, 0u, 0u, 0u);
        const uint64_t opaque = __ballot(lane < n && l_src[w][lane].w == kInvN);
        uint32_t t = transpose32(mine.x);
        uint64_t L = (uint64_t)(uint32_t)__shfl((int)t, cell, 64) | ((uint64_t)(uint32_t)__shfl((int)t, 32 + cell, 64) << 32);
        if (x >= W) L = 0ull;
        if (opaque) {
            t = transpose32(mine.y);
            const uint64_t E =
                (uint64_t)(uint32_t)__shfl((int)t, cell, 64) | ((uint64_t)(uint32_t)__shfl((int)t, 32 + cell, 64) << 32);
            const uint64_t T = L & ~E & opaque;
            if (T) L &= ~0ull << (63 - (int)__builtin_clzll(T));
        }
        // the next bucket of the lane's column and its sample counts, a pass ahead
        int b = 0;
        uint32_t cnt = kFull;
        auto next = [&]() {
            b = (int)__builtin_ctzll(L);
            const uint2 e = *(const uint2 *)&l_ent[w][b].y;
            cnt = kFull;
            if ((e.x >> cell) & 1u) cnt = A.icov[e.y + (uint32_t)__popc(e.x & ((1u << cell) - 1u))] >> half;
        };
        if (L) next();
        while (__ballot(L != 0ull)) {
            // gradient paints cost several solid ones: they wait until no lane has a solid
            // paint next, and are then blended by all lanes that hold one
            bool turn = L != 0ull;
            if (GRAD) {
                const bool solid = turn && l_src[w][b].w >= 0.f;
                if (__ballot(solid)) {
                    turn = solid;
                } else {
                    if (turn) {
                        const float4 src = l_src[w][b];
                        const uint32_t c = __float_as_uint(src.x);
                        int ix0, iw;
                        item_extent(A.prec, src, l_ent[w][b], cell, tx0, ix0, iw);
                        const float4 p0 = grad_color(A.G, c, ix0, iw, x, 2 * r, s_dec, s_deca);
                        const float4 p1 = grad_color(A.G, c, ix0, iw, x, 2 * r + 1, s_dec, s_deca);
                        blend_dec<SRGB>(s_step, d0, p0, p0.w * ((float)(cnt & 63u) * kInvN));
                        blend_dec<SRGB>(s_step, d1, p1, p1.w * ((float)((cnt >> 6) & 63u) * kInvN));
                        L &= L - 1ull;
                        if (L) next();
                    }
                    continue;
                }
            }
            if (turn) {
                const float4 src = l_src[w][b];
                const uint32_t cc = cnt;
                L &= L - 1ull;
                if (L) next();
                blend_dec<SRGB>(s_step, d0, src, src.w * (float)(cc & 63u));
                blend_dec<SRGB>(s_step, d1, src, src.w * (float)((cc >> 6) & 63u));
            }
        }
        wave_sync_lds();
    };

    const uint32_t q0 = A.rowstart[row0 + r], q1 = A.rowstart[row0 + r + 1];
    list_row<GRAD>(A, q0, q1, tx, tx1, kInvN, s_dec, l_queue[w], l_src[w], l_ent[w], flush);

    if (x >= W) return;
    const int y0 = 2 * r;
    *(uint32_t *)(image + (size_t)y0 * pitch + (size_t)x * 4) = pack_dec<SRGB>(s_step, d0);
    if (y0 + 1 < H) *(uint32_t *)(image + (size_t)(y0 + 1) * pitch + (size_t)x * 4) = pack_dec<SRGB>(s_step, d1);
}

// ---------------------------------------------------------------------------------
// multisample compositor (ms_output_{8,32}.frag.glsl: every covered sample of an N-sample
// 8-bit framebuffer is blended src-over and re-quantised; ras_base.cpp:1148-1163 then
// resolves each pixel to the average of its samples' decoded values, summed in sample
// order).  The bucket lookup is the coverage compositor's (lane = pixel column); the
// blending runs with lane = sample: lane q * 2N + dy * N + s holds sample s of pixel
// (column p * CPR + q, row 2r + dy) of the 64x2 tile in state register p, CPR = 64 / 2N
// columns per register.  Each register that holds a pixel covered by the bucket costs one
// wave-wide blend (its lanes select by their sample bits), so a 2x2 fragment or a span
// column costs the same whatever its sample count, and no lane loops over samples.  Solid
// paints run over the state registers in static blocks of four registers at 32 samples,
// two at 16 and 8 (apply_blocks): a register's blend is four byte lookups in the path's
// table and one select whose lane mask is read straight from the column lanes' sample
// bits, with no register indexing.
// ---------------------------------------------------------------------------------
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));

// Runs f(state, p) -> new state on every register of the BLK-register blocks of vec that
// hold a set bit of m (p = pbase + register), with static register numbers: the state
// stays in plain VGPRs (no indexing, no per-register loop), and a block's LDS round trips
// overlap, at the price of the block's uncovered registers (f leaves a register it does not
// cover unchanged).
template <int N, int BLK, class V, class F>
__device__ __forceinline__ void apply_blocks(V &vec, uint32_t m, int pbase, const F &f) {
#pragma unroll
    for (int b0 = 0; b0 < N; b0 += BLK) {
        if ((m >> b0) & ((1u << BLK) - 1u)) {
#pragma unroll
            for (int i = 0; i < BLK; ++i) vec[b0 + i] = f(vec[b0 + i], pbase + b0 + i);
        }
    }
}

// Runs f(state, p) -> new state on every register p of the set bits of m (p = pbase + bit)
// by index: the register number is wave-uniform, so the indexed state stays in VGPRs
// (s_set_gpr_idx).  The gradient variants use these, since their paint arithmetic per
// register is large (the static blocks would spend it on uncovered registers too) and a
// function that mixes indexed and static access to the state spills it.  The 4-way form
// takes four registers an iteration so that their LDS round trips overlap; missing ones
// repeat the first register, whose duplicate writes store the same value, so every write
// is unconditional.  A write that depends on control flow inside the loop makes the
// compiler copy the whole 32-register vector at every iteration, and so does a loop that
// writes two vectors: each call covers one.
template <class V, class F>
__device__ __forceinline__ void apply_regs4(V &vec, uint32_t m, int pbase, const F &f) {
    while (m) {
        const int c0 = __builtin_amdgcn_readfirstlane((int)__builtin_ctz(m));
        m &= m - 1u;
        const int c1 = m ? __builtin_amdgcn_readfirstlane((int)__builtin_ctz(m)) : c0;
        m &= m - 1u;
        const int c2 = m ? __builtin_amdgcn_readfirstlane((int)__builtin_ctz(m)) : c0;
        m &= m - 1u;
        const int c3 = m ? __builtin_amdgcn_readfirstlane((int)__builtin_ctz(m)) : c0;
        m &= m - 1u;
        const uint32_t o0 = vec[c0], o1 = vec[c1], o2 = vec[c2], o3 = vec[c3];
        const uint32_t n0 = f(o0, pbase + c0), n1 = f(o1, pbase + c1), n2 = f(o2, pbase + c2),
                       n3 = f(o3, pbase + c3);
        vec[c3] = n3;
        vec[c2] = n2;
        vec[c1] = n1;
        vec[c0] = n0;
    }
}

template <class V, class F>
__device__ __forceinline__ void apply_regs1(V &vec, uint32_t m, int pbase, const F &f) {
    while (m) {
        const int c = __builtin_amdgcn_readfirstlane((int)__builtin_ctz(m));
        m &= m - 1u;
        vec[c] = f(vec[c], pbase + c);
    }
}

template <int NREG> struct SampleRegs;
template <> struct SampleRegs<64> {
    u32x32 a, b;
    __device__ __forceinline__ void init(uint32_t v) {
#pragma unroll
        for (int i = 0; i < 32; ++i) { a[i] = v; b[i] = v; }
    }
    __device__ __forceinline__ uint32_t get(int p) const { return p < 32 ? a[p] : b[p - 32]; }
    template <int BLK, class F> __device__ __forceinline__ void apply(uint64_t m, const F &f) {
        apply_blocks<32, BLK>(a, (uint32_t)m, 0, f);
        apply_blocks<32, BLK>(b, (uint32_t)(m >> 32), 32, f);
    }
    template <class F> __device__ __forceinline__ void apply4(uint64_t m, const F &f) {
        apply_regs4(a, (uint32_t)m, 0, f);
        apply_regs4(b, (uint32_t)(m >> 32), 32, f);
    }
    template <class F> __device__ __forceinline__ void apply1(uint64_t m, const F &f) {
        apply_regs1(a, (uint32_t)m, 0, f);
        apply_regs1(b, (uint32_t)(m >> 32), 32, f);
    }
};
template <> struct SampleRegs<32> {
    u32x32 a;
    __device__ __forceinline__ void init(uint32_t v) {
#pragma unroll
        for (int i = 0; i < 32; ++i) a[i] = v;
    }
    __device__ __forceinline__ uint32_t get(int p) const { return a[p]; }
    template <int BLK, class F> __device__ __forceinline__ void apply(uint64_t m, const F &f) {
        apply_blocks<32, BLK>(a, (uint32_t)m, 0, f);
    }
    template <class F> __device__ __forceinline__ void apply4(uint64_t m, const F &f) { apply_regs4(a, (uint32_t)m, 0, f); }
    template <class F> __device__ __forceinline__ void apply1(uint64_t m, const F &f) { apply_regs1(a, (uint32_t)m, 0, f); }
};
template <> struct SampleRegs<16> {
    u32x16 a;
    __device__ __forceinline__ void init(uint32_t v) {
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] = v;
    }
    __device__ __forceinline__ uint32_t get(int p) const { return a[p]; }
    template <int BLK, class F> __device__ __forceinline__ void apply(uint64_t m, const F &f) {
        apply_blocks<16, BLK>(a, (uint32_t)m, 0, f);
    }
    template <class F> __device__ __forceinline__ void apply4(uint64_t m, const F &f) { apply_regs4(a, (uint32_t)m, 0, f); }
    template <class F> __device__ __forceinline__ void apply1(uint64_t m, const F &f) { apply_regs1(a, (uint32_t)m, 0, f); }
};

// Blend tables of the solid paints, one per path, built once per frame: byte ch * 256 + k
// of a path's 1 KiB table holds the code that channel ch takes when the path's paint
// (decoded colour, alpha a) is blended over code k -- blend_code's arithmetic per channel.
// Lane l of a path's wave computes codes 4l .. 4l + 3 of every channel.  Words without
// alpha (gradients, no paint) get no table.
template <bool SRGB>
__global__ void __launch_bounds__(256) k_paint_tables(uint32_t P, const uint32_t *__restrict__ finfo,
                                                      const float *__restrict__ dec, const float4 *__restrict__ step,
                                                      uint32_t *__restrict__ ptab) {
    const uint32_t path = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (path >= P) return;
    const uint32_t c = finfo[path];
    if (!(c & 0xFF000000u)) return;
    const int lane = threadIdx.x & 63;
    const float4 src = make_float4(dec[c & 0xFFu], dec[(c >> 8) & 0xFFu], dec[(c >> 16) & 0xFFu], unorm_dec((int)(c >> 24)));
    const float a = src.w, oma = 1.f - a;
    uint32_t e[4];  // e[ch]: channel ch's codes for k = 4l .. 4l + 3, one byte each
    e[0] = e[1] = e[2] = e[3] = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k = 4 * lane + j;
        const float dk = SRGB ? dec[k] : unorm_dec(k);
        const float v0 = src.x * a + dk * oma;
        const float v1 = src.y * a + dk * oma;
        const float v2 = src.z * a + dk * oma;
        const float va = a * a + unorm_dec(k) * oma;
        float t;
        const uint32_t c0 = SRGB ? (uint32_t)srgb_code(step, v0, t) : (uint32_t)unorm_code(v0);
        const uint32_t c1 = SRGB ? (uint32_t)srgb_code(step, v1, t) : (uint32_t)unorm_code(v1);
        const uint32_t c2 = SRGB ? (uint32_t)srgb_code(step, v2, t) : (uint32_t)unorm_code(v2);
        e[0] |= c0 << (8 * j);
        e[1] |= c1 << (8 * j);
        e[2] |= c2 << (8 * j);
        e[3] |= (uint32_t)unorm_code(va) << (8 * j);
    }
    uint32_t *t = ptab + (size_t)path * 256;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) t[ch * 64 + lane] = e[ch];
}

// A code's blend through a planar table: channel ch's byte indexes bytes ch * 256 .. +255.
__device__ __forceinline__ uint32_t table_code(const uint32_t *T, uint32_t st) {
    const uint8_t *b = (const uint8_t *)T;
    const uint32_t lo = (uint32_t)b[st & 0xFFu] | ((uint32_t)b[256 + ((st >> 8) & 0xFFu)] << 8);
    const uint32_t hi = (uint32_t)b[512 + ((st >> 16) & 0xFFu)] | ((uint32_t)b[768 + (st >> 24)] << 8);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);  // the low half-words of lo and hi
}

// One sample's framebuffer code blended with paint src (decoded colour, alpha a) and
// re-quantised: the arithmetic of blend_dec on the decoded code.
template <bool SRGB>
__device__ __forceinline__ uint32_t blend_code(const float4 *step, const float *dec, uint32_t code,
                                               const float4 &src, float a) {
    const float oma = 1.f - a;
    const uint32_t k0 = code & 0xFFu, k1 = (code >> 8) & 0xFFu, k2 = (code >> 16) & 0xFFu;
    const float d0 = SRGB ? dec[k0] : unorm_dec((int)k0);
    const float d1 = SRGB ? dec[k1] : unorm_dec((int)k1);
    const float d2 = SRGB ? dec[k2] : unorm_dec((int)k2);
    const float da = unorm_dec((int)(code >> 24));
    const float v0 = src.x * a + d0 * oma;
    const float v1 = src.y * a + d1 * oma;
    const float v2 = src.z * a + d2 * oma;
    const float va = a * a + da * oma;
    float t;
    const uint32_t c0 = SRGB ? (uint32_t)srgb_code(step, v0, t) : (uint32_t)unorm_code(v0);
    const uint32_t c1 = SRGB ? (uint32_t)srgb_code(step, v1, t) : (uint32_t)unorm_code(v1);
    const uint32_t c2 = SRGB ? (uint32_t)srgb_code(step, v2, t) : (uint32_t)unorm_code(v2);
    return c0 | (c1 << 8) | (c2 << 16) | ((uint32_t)unorm_code(va) << 24);
}

// Bit i of the result is set when any of bits [i * CPR, (i + 1) * CPR) of e is.
template <int CPR>
__device__ __forceinline__ uint64_t group_bits(uint64_t e) {
    if (CPR == 1) return e;
    if (CPR == 2) {
        uint64_t x = (e | (e >> 1)) & 0x5555555555555555ull;
        x = (x | (x >> 1)) & 0x3333333333333333ull;
        x = (x | (x >> 2)) & 0x0F0F0F0F0F0F0F0Full;
        x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
        x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
        return (x | (x >> 16)) & 0xFFFFFFFFull;
    }
    uint64_t x = (e | (e >> 1) | (e >> 2) | (e >> 3)) & 0x1111111111111111ull;
    x = (x | (x >> 3)) & 0x0303030303030303ull;
    x = (x | (x >> 6)) & 0x000F000F000F000Full;
    x = (x | (x >> 12)) & 0x000000FF000000FFull;
    return (x | (x >> 24)) & 0xFFFFull;
}

// The sample bits of the two pixels of column offset dx in a merged mask (the reference's
// layout: N = 8 one byte per pixel (dx * 2 + dy), N = 16 one half-word per pixel in word dx,
// N = 32 one word per pixel dx * 2 + dy): row 0 in the low N bits, row 1 above (N = 32:
// row 1 in `hi`).
template <int SPP>
__device__ __forceinline__ uint32_t column_bits(const uint32_t *m, int dx, uint32_t &hi) {
    if (SPP == 32) {
        hi = dx ? m[3] : m[1];
        return dx ? m[2] : m[0];
    }
    hi = 0u;
    if (SPP == 16) return dx ? m[1] : m[0];
    return (m[0] >> (16 * dx)) & 0xFFFFu;
}

// Measured on the headline scene's multisample composite at 32 / 16 / 8 samples: the
// static blocks take 10.0 / 5.6 / 4.15 ms where the indexed four-register loop took
// 13.9 / 7.4 / 4.6 ms (per register it spent 14 VALU, 9 scalar and 5 LDS instructions
// against 10 VALU and 4 LDS, the blocks' idle registers included).  At 32 samples, blocks
// of two or eight registers, one- or four-bucket groups, and three or five waves per SIMD
// were all slower (10.2 / 10.3 / 10.6 / 10.5 / 11.7 / 15.1 ms: five waves spill 176 bytes
// a lane); blocks of four cost 5.7 / 4.3 ms at 16 / 8 samples.  Two buckets a group with
// registers capped for 4 / 5 / 7 waves per SIMD at 32 / 16 / 8 samples (16 bytes a lane
// spilled at 32; six waves at 16 samples: 6.0 ms, eight at 8: 4.6 ms).
// The gradient variants, whose paint arithmetic would spill under those caps, take four-bucket
// groups, the indexed loops and 3 / 4 / 4 waves.  What they read besides a pixel's own values
// is kept out of the registers' loop: the covering item's extent is looked up once a column,
// and the gradient's word is one for the wave, so its table comes by scalar loads.  1024x1024,
// 800 gradient paths, 32 / 16 / 8 samples: 7.2 / 3.5 / 1.88 ms, with the look-up in the loop,
// vector loads and 40 KB of LDS exceeded (a wave less each) 8.9 / 4.2 / 2.30; groups of two
// 7.3 / 3.7 / 1.90 and a quarter slower on glyphs at 32 samples, of eight 8.8 / 4.7 / 2.58,
// five waves at 16 and 8 samples 3.6 / 1.91 and a fifth slower on small canvases.
template <int SPP, bool SRGB, bool GRAD>
__global__ void __launch_bounds__(256, GRAD ? (SPP == 32 ? 3 : 4) : (SPP == 32 ? 4 : (SPP == 16 ? 5 : 7))) k_composite_ms(CovArgs A) {
    constexpr int NW = Words<SPP>::n;
    constexpr int CPR = 64 / (2 * SPP);
    constexpr int NREG = 64 / CPR;
    constexpr int G = GRAD ? 4 : 2;
    constexpr uint32_t FULL = SPP == 8 ? 0xFFFFu : 0xFFFFFFFFu;  // both rows' bits (N = 32: each row)
    __shared__ float4 s_step[SRGB && GRAD ? kQuantSteps : 1];
    __shared__ float s_dec[256];
    __shared__ float s_deca[GRAD ? 256 : 1];
    __shared__ float4 l_src[4][kCovList];
    __shared__ uint4 l_ent[4][kCovList];
    __shared__ uint32_t l_queue[4][kRowQueue];
    __shared__ uint32_t tbl[4][G][256];     // the paths' blend tables; then the final average's staging
    for (int i = threadIdx.x; i < 256; i += 256) {
        s_dec[i] = A.dec_c[i];
        if (GRAD) s_deca[i] = A.dec_a[i];
    }
    for (int i = threadIdx.x; i < (SRGB && GRAD ? kQuantSteps : 0); i += 256) s_step[i] = A.step_c[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int W = A.W, H = A.H, tiles_x = A.tiles_x;
    // XCD-aware tile order of the coverage compositor: XCD b % 8 takes whole cell rows
    const int xcd = (int)(blockIdx.x & 7u), t = (int)(blockIdx.x >> 3) * 4 + w;
    const int rr = t / tiles_x, r = xcd + 8 * rr;
    if (r >= (H + 1) / 2) return;
    const int tx = t - rr * tiles_x, tx0 = tx * 64;
    const int tx1 = tmin(tx0 + 64, W);
    const int x = tx0 + lane, cell = lane >> 1;
    // blend-phase coordinates of this lane
    const int q = lane / (2 * SPP), dy = (lane / SPP) & 1;
    SampleRegs<NREG> S;
    S.init(0xFFFFFFFFu);

    auto flush = [&](int nlist) {
        wave_sync_lds();
        for (int g0 = 0; g0 < nlist; g0 += G) {
            const int ng = tmin(G, nlist - g0);
            uint4 tv[G];
            // per column (lane): the sample bits of both rows under each bucket's covering
            // item, 0 where no item covers it
            uint32_t cb[G], cbh[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint4 e = g < ng ? l_ent[w][g0 + g] : make_uint4(0u, 0u, 0u, 0u);
                // the path's blend table (solid paints; a gradient's l_src.w is negative)
                const bool solid = g < ng && !(GRAD && l_src[w][g0 + g].w < 0.f);
                tv[g] = solid ? *(const uint4 *)(A.ptab + (size_t)e.w * 256 + 4 * lane) : make_uint4(0u, 0u, 0u, 0u);
                cb[g] = cbh[g] = 0u;
                if (((e.x >> cell) & 1u) && x < W) {
                    uint32_t hi = FULL, lo = FULL;
                    if ((e.y >> cell) & 1u) {
                        uint32_t pm[NW];
                        load_mask<NW>(A.imask, (size_t)e.z + (uint32_t)__popc(e.y & ((1u << cell) - 1u)), pm);
                        lo = column_bits<SPP>(pm, lane & 1, hi);
                    }
                    cb[g] = lo;
                    cbh[g] = SPP == 32 ? hi : 0u;
                }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) *(uint4 *)&tbl[w][g][4 * lane] = tv[g];
            wave_sync_lds();
            // blend, bucket by bucket in path order, one wave-wide pass per state register
            // holding a covered column: four LDS reads of the path's blend table for a
            // solid paint, the blend arithmetic on the pixel's own paint for a gradient.
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (g >= ng) break;
                const uint64_t regs = group_bits<CPR>(__ballot((cb[g] | cbh[g]) != 0u));
                if (!regs) continue;
                const float4 src = l_src[w][g0 + g];
                const bool gpaint = GRAD && src.w < 0.f;
                // register p's lanes are its columns' sample bits in column order (lane
                // q * 2N + dy * N + s is bit dy * N + s of column p * CPR + q; N = 32: the
                // rows' words cb, cbh), so the covered lanes form one wave-wide mask read
                // from the columns' lanes -- the select takes it as a lane mask directly
                const uint32_t cbg = cb[g], cbhg = cbh[g];
                auto covers = [&](int p) -> bool {
                    uint64_t m;
                    if (SPP == 32) {
                        m = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)cbg, p) |
                            ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)cbhg, p) << 32);
                    } else {
                        m = 0ull;
#pragma unroll
                        for (int k = 0; k < CPR; ++k)
                            m |= (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)cbg, p * CPR + k) << (2 * SPP * k);
                    }
                    return __builtin_amdgcn_inverse_ballot_w64(m);
                };
                if (!gpaint) {
                    auto blend = [&](uint32_t st, int p) -> uint32_t {
                        const uint32_t nst = table_code(tbl[w][g], st);
                        return covers(p) ? nst : st;
                    };
                    if (GRAD) S.apply4(regs, blend);
                    else S.template apply<SPP == 32 ? 4 : 2>(regs, blend);
                } else {
                    // the covering item's extent, once a column
                    const uint4 e = l_ent[w][g0 + g];
                    int ix0 = 0, iw = 1;
                    if ((e.x >> cell) & 1u) item_extent(A.prec, src, e, cell, tx0, ix0, iw);
                    const uint32_t ce = (uint32_t)ix0 | ((uint32_t)iw << 16);
                    const uint32_t word = (uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(src.x));
                    S.apply1(regs, [&](uint32_t st, int p) -> uint32_t {
                        const int c = p * CPR + q;
                        const uint32_t ext = (uint32_t)__shfl((int)ce, c, 64);
                        const float4 pa = grad_color(A.G, word, (int)(ext & 0xFFFFu), (int)(ext >> 16),
                                                     tx0 + c, 2 * r + dy, s_dec, s_deca);
                        const uint32_t nst = blend_code<SRGB>(s_step, s_dec, st, pa, pa.w);
                        return covers(p) ? nst : st;
                    });
                }
            }
            wave_sync_lds();
        }
    };

    const uint32_t q0 = A.rowstart[r], q1 = A.rowstart[r + 1];
    list_row<GRAD>(A, q0, q1, tx, tx1, 1.f, s_dec, l_queue[w], l_src[w], l_ent[w], flush);

    // resolve: G registers at a time are staged in this wave's tables (G x 64 words);
    // lane (pixel, channel) sums the pixel's decoded samples in sample order, divides by N
    // and re-quantises, and the four channel lanes of a pixel assemble its word
    static_assert(NREG % G == 0, "state registers are staged G at a time");
    uint32_t *stg = &tbl[w][0][0];
    wave_sync_lds();
#pragma unroll
    for (int p0 = 0; p0 < NREG; p0 += G) {
#pragma unroll
        for (int k = 0; k < G; ++k) stg[k * 64 + lane] = S.get(p0 + k);
        wave_sync_lds();
#pragma unroll
        for (int t0 = 0; t0 < 8 * G * CPR; t0 += 64) {
            const int tt = t0 + lane;
            const int ch = tt & 3, pix = tt >> 2;           // pix = (k * CPR + qq) * 2 + row, k < G
            const int row = pix & 1, kq = pix >> 1, k = kq / CPR, qq = kq - k * CPR;
            const bool live = tt < 8 * G * CPR;
            const uint32_t *smps = stg + k * 64 + qq * 2 * SPP + row * SPP;
            float sum = 0.f;
            if (live) {
#pragma unroll 8
                for (int s2 = 0; s2 < SPP; ++s2) {
                    const uint32_t b = (smps[s2] >> (8 * ch)) & 0xFFu;
                    sum += (SRGB && ch < 3) ? s_dec[b] : unorm_dec((int)b);
                }
            }
            const float avg = sum / (float)SPP;
            float tmp;
            const uint32_t code = (SRGB && ch < 3) ? (uint32_t)srgb_code(GRAD ? s_step : A.step_c, avg, tmp) : (uint32_t)unorm_code(avg);
            uint32_t word = code << (8 * ch);
            word |= (uint32_t)__shfl_xor((int)word, 1, 64);
            word |= (uint32_t)__shfl_xor((int)word, 2, 64);
            const int col = tx0 + (p0 + k) * CPR + qq, y = 2 * r + row;
            if (live && ch == 0 && col < W && y < H) *(uint32_t *)(A.image + (size_t)y * A.pitch + (size_t)col * 4) = word;
        }
        wave_sync_lds();
    }
}

// Device requantisation of arbitrary values (colour-table self-check): codes and the
// decoded values of the codes.
template <bool SRGB>
__global__ void k_encode_values(int64_t n, const float *__restrict__ v, const float4 *__restrict__ step,
                                uint8_t *__restrict__ code, float *__restrict__ dec) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float d;
    int k;
    if (SRGB) {
        k = srgb_code(step, v[i], d);
    } else {
        k = unorm_code(v[i]);
        d = unorm_dec(k);
    }
    code[i] = (uint8_t)k;
    dec[i] = d;
}

// Exhaustive comparison of the device requantisation with the threshold tables over every
// float bit pattern in [lo, hi): counts disagreements of code or decoded value.
template <bool SRGB>
__global__ void k_encode_sweep(uint32_t lo, uint32_t hi, const float4 *__restrict__ step,
                               const float *__restrict__ thr, const float *__restrict__ dec, unsigned long long *bad) {
    unsigned long long nbad = 0;
    for (uint64_t b = (uint64_t)lo + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; b < hi;
         b += (uint64_t)gridDim.x * blockDim.x) {
        const float v = __uint_as_float((uint32_t)b);
        int ref = 0;
#pragma unroll 1
        for (int s = 128; s >= 1; s >>= 1)
            if (ref + s <= 255 && v >= thr[ref + s]) ref += s;
        float d;
        int k;
        if (SRGB) {
            k = srgb_code(step, v, d);
        } else {
            k = unorm_code(v);
            d = unorm_dec(k);
        }
        nbad += (k != ref || __float_as_uint(d) != __float_as_uint(dec[ref])) ? 1ull : 0ull;
    }
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) nbad += __shfl_xor(nbad, dd, 64);
    if ((threadIdx.x & 63) == 0 && nbad) atomicAdd(bad, nbad);
}

// draw list + merged masks in the reference's order and layout (.cu:789-868, 1195-1266)
template <int SPP>
__global__ void k_debug_draw(int64_t NB, const int2 *__restrict__ binfo, const uint32_t *__restrict__ finfo,
                             const uint32_t *__restrict__ boff, const uint2 *__restrict__ bcnt,
                             const uint32_t *__restrict__ items, const uint32_t *__restrict__ imask,
                             const uint32_t *__restrict__ moff, const uint32_t *__restrict__ ioff, int4 *draw,
                             uint32_t *mmask4) {
    constexpr int NW = Words<SPP>::n;
    int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= NB) return;
    const uint32_t cnt = bcnt[b].x;
    if (!cnt) return;
    const int2 info = binfo[b];
    const uint32_t fill = finfo[info.x];
    const int y = 2 * info.y;
    const size_t ib = 2 * (size_t)boff[b];
    uint32_t mi = moff[b];
    const uint32_t io = ioff[b];
    uint32_t o = io;
    size_t mj = boff[b];  // the bucket's merged cells' masks, in x order
    auto put_merged = [&](int x0) {
        draw[o++] = make_int4((int32_t)(((uint32_t)y << 16) | (uint32_t)x0), 2, (int)fill, (int)(mi + 1));
        uint32_t mk[4] = {0u, 0u, 0u, 0u};
        load_mask<NW>(imask, mj++, mk);
        *(uint4 *)(mmask4 + 4 * (size_t)mi) = make_uint4(mk[0], mk[1], mk[2], mk[3]);
        ++mi;
    };
    for (uint32_t j = 0; j < cnt; ++j) {
        const uint32_t it = items[ib + j];
        const int x0 = (int)(it & 0xFFFFu), w = (int)(it >> 16);
        if (w == 0) {
            put_merged(x0);
            continue;
        }
        // a span followed by the merged fragment it ends at: the reference emits that
        // fragment first (.cu:836-862)
        const bool pair = j + 1 < cnt && (items[ib + j + 1] >> 16) == 0u &&
                          (int)(items[ib + j + 1] & 0xFFFFu) == x0 + w;
        if (pair) put_merged(x0 + w);
        draw[o++] = make_int4((int32_t)(((uint32_t)y << 16) | (uint32_t)x0), w, (int)fill, 0);
        if (pair) ++j;
    }
}

// out[0] += merged cells, out[1] += items
__global__ void __launch_bounds__(256) k_count_reduce(const uint2 *__restrict__ bcnt, size_t n, unsigned long long *out) {
    __shared__ unsigned long long part[2][4];
    unsigned long long sa = 0, sc = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint2 c = bcnt[i];
        sa += c.y;
        sc += c.x;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        sa += __shfl_xor(sa, d, 64);
        sc += __shfl_xor(sc, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = sa;
        part[1][threadIdx.x >> 6] = sc;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const unsigned long long t = part[threadIdx.x][0] + part[threadIdx.x][1] + part[threadIdx.x][2] + part[threadIdx.x][3];
        atomicAdd(&out[threadIdx.x], t);
    }
}

__global__ void k_debug_counts(int64_t NB, const uint2 *__restrict__ bcnt, uint32_t *merged, uint32_t *items) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= NB) return;
    merged[b] = bcnt[b].y;
    items[b] = bcnt[b].x;
}

inline unsigned blocks_for(int64_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

void launch_resolve(const SceneDev &sc, const Tables &t, Frame &f, hipStream_t s) {
    if (!f.NB) return;
    ResolveArgs A;
    A.NB = f.NB; A.binfo = f.binfo; A.boff = f.boff; A.bcarry = f.bcarry; A.frule = sc.frule;
    A.rec = f.rec; A.F = f.F; A.scratch = f.scratch_keys; A.W = f.W;
    A.pcanvas = sc.pcanvas; A.scarry = f.scarry;
    // the merged masks feed the multisample compositor and the debug draw list; the
    // coverage compositor reads only the per-pixel sample counts
    A.items = f.items; A.imask = f.imask; A.icov = f.icov; A.prec = f.prec;
    A.rpos = f.rpos; A.finfo = sc.finfo; A.rext = f.rext; A.rrec = f.rrec; A.rtile = f.rtile; A.bcnt = f.bcnt;
    A.big_list = f.big_list; A.big_count = f.big_count;
    // A wave resolves up to 64 buckets of the grid's stride: with fewer its packs of four and two
    // small buckets stay part empty and every bucket pays for a wave's start and end.  One bucket
    // a wave up to 65536 waves, then shared / this, us: 47 k buckets 42 / 22, 57 k (a page of
    // text) 62 / 32, a poster 152 / 107, 1.9 M 434 / 426, 1.8 M (the illustration) 1325 / 1304;
    // at most 96 buckets 438 and 1364.  The least number of waves weighs small frames, which
    // lose by waves of fewer buckets, against middling ones, whose uneven buckets balance over
    // two turns of the 5120 resident waves.  Stage with at least 5120 / 7680 / 10240, us: 512x512,
    // 200 paths 26 / 28 / 28, the page 34 / 38 / 37, 1000x1000, 300 paths 58 / 58 / 59; 1024x768,
    // 1500 paths 175 / 172 / 165, 1000x777, 2000 paths 300 / 309 / 276, 1279x719, 3000 paths
    // 177 / 177 / 171, 2048x2048, 20000 glyphs 123 / 114 / 111, 1500x1500, 6000 paths
    // 456 / 455 / 437.
    const int64_t gd = std::max((f.NB + 63) / 64, kResolveWaves);
    const unsigned g1 = (unsigned)std::min<int64_t>(f.NB, f.resolve_grid > 0 ? f.resolve_grid : gd);
    const unsigned gc = f.class_grid > 0 ? (unsigned)f.class_grid : 4096u;
    dim3 b64(64);
#define SL_LAUNCH2(N, K)                                                              \
    do {                                                                              \
        hipLaunchKernelGGL((k_resolve_first<N, K>), dim3(g1), b64, 0, s, A);          \
        hipLaunchKernelGGL((k_resolve_big<N, K>), dim3(gc), dim3(kBigThreads), 0, s, A); \
        hipLaunchKernelGGL((k_resolve_huge<N, K>), dim3(1024), dim3(kBigThreads), 0, s, A); \
    } while (0)
#define SL_LAUNCH(N)                                                                  \
    do {                                                                              \
        if (f.keep_masks) SL_LAUNCH2(N, true);                                        \
        else SL_LAUNCH2(N, false);                                                    \
    } while (0)
    if (t.spp == 8) SL_LAUNCH(8);
    else if (t.spp == 16) SL_LAUNCH(16);
    else SL_LAUNCH(32);
#undef SL_LAUNCH
}

void launch_scene_carry(const SceneDev &sc, Frame &f, hipStream_t s) {
    (void)sc;
    if (!f.nscenes) return;
    hipLaunchKernelGGL(k_scene_carry, dim3(blocks_for(f.nscenes, 256)), dim3(256), 0, s, f.nscenes, f.sfirst,
                       (const uint32_t *)f.pbase, (const uint32_t *)f.bcarry, f.scarry);
}

void launch_composite(const SceneDev &sc, const Tables &t, Frame &f, hipStream_t s) {
    const int R = (f.H + 1) / 2;
    const int tiles_x = (f.W + 63) / 64;
    const int64_t ntiles = f.nscenes ? f.ntiles : (int64_t)R * tiles_x;
    if (!f.ms) {
        CovArgs C;
        C.W = f.W; C.H = f.H; C.tiles_x = tiles_x;
        C.rowstart = f.rowstart; C.rext = f.rext; C.rrec = f.rrec; C.rtile = f.rtile;
        C.prec = f.prec; C.icov = f.icov; C.imask = nullptr; C.ptab = nullptr; C.dec_c = t.dec_c; C.dec_a = t.dec_a; C.step_c = t.step_c;
        C.image = f.image; C.pitch = f.pitch;
        C.G = f.grad;
        C.nscenes = f.nscenes; C.ntiles = ntiles; C.stile = f.stile; C.simg = f.simg;
        // one scene: 8 XCD row sets of ceil(R / 8) rows each; a batch: tiles in order
        dim3 g(f.nscenes ? blocks_for(ntiles, 4) : 8u * blocks_for((int64_t)tiles_x * ((R + 7) / 8), 4)), b(256);
#define SL_LAUNCH(N, SR)                                                                   \
    do {                                                                                   \
        if (f.nscenes) hipLaunchKernelGGL((k_composite_cov<N, SR, true, false>), g, b, 0, s, C);        \
        else if (f.has_grad) hipLaunchKernelGGL((k_composite_cov<N, SR, false, true>), g, b, 0, s, C);  \
        else hipLaunchKernelGGL((k_composite_cov<N, SR, false, false>), g, b, 0, s, C);                 \
    } while (0)
        if (f.srgb) {
            if (t.spp == 8) SL_LAUNCH(8, true);
            else if (t.spp == 16) SL_LAUNCH(16, true);
            else SL_LAUNCH(32, true);
        } else {
            if (t.spp == 8) SL_LAUNCH(8, false);
            else if (t.spp == 16) SL_LAUNCH(16, false);
            else SL_LAUNCH(32, false);
        }
#undef SL_LAUNCH
        return;
    }
    CovArgs C;
    C.W = f.W; C.H = f.H; C.tiles_x = tiles_x;
    C.rowstart = f.rowstart; C.rext = f.rext; C.rrec = f.rrec; C.rtile = f.rtile;
    C.prec = f.prec; C.icov = f.icov; C.imask = f.imask; C.ptab = f.ptab;
    C.dec_c = t.dec_c; C.dec_a = t.dec_a; C.step_c = t.step_c;
    C.image = f.image; C.pitch = f.pitch;
    C.G = f.grad;
    C.nscenes = 0; C.ntiles = ntiles; C.stile = nullptr; C.simg = nullptr;
    if (sc.P) {
        if (f.srgb)
            hipLaunchKernelGGL(k_paint_tables<true>, dim3(blocks_for(sc.P, 4)), dim3(256), 0, s, (uint32_t)sc.P, sc.finfo,
                               t.dec_c, t.step_c, f.ptab);
        else
            hipLaunchKernelGGL(k_paint_tables<false>, dim3(blocks_for(sc.P, 4)), dim3(256), 0, s, (uint32_t)sc.P, sc.finfo,
                               t.dec_c, t.step_c, f.ptab);
    }
    dim3 g(8u * blocks_for((int64_t)tiles_x * ((R + 7) / 8), 4)), b(256);
#define SL_LAUNCH(N)                                                                                    \
    do {                                                                                                \
        if (f.has_grad) {                                                                               \
            if (f.srgb) hipLaunchKernelGGL((k_composite_ms<N, true, true>), g, b, 0, s, C);             \
            else hipLaunchKernelGGL((k_composite_ms<N, false, true>), g, b, 0, s, C);                   \
        } else {                                                                                        \
            if (f.srgb) hipLaunchKernelGGL((k_composite_ms<N, true, false>), g, b, 0, s, C);            \
            else hipLaunchKernelGGL((k_composite_ms<N, false, false>), g, b, 0, s, C);                  \
        }                                                                                               \
    } while (0)
    if (t.spp == 8) SL_LAUNCH(8);
    else if (t.spp == 16) SL_LAUNCH(16);
    else SL_LAUNCH(32);
#undef SL_LAUNCH
}

void launch_encode_values(const Tables &t, int channel, const float *v, int64_t n, uint8_t *code, float *dec,
                          hipStream_t s) {
    if (n <= 0) return;
    dim3 g(blocks_for(n, 256)), b(256);
    if (channel == 0 && t.srgb)
        hipLaunchKernelGGL(k_encode_values<true>, g, b, 0, s, n, v, t.step_c, code, dec);
    else
        hipLaunchKernelGGL(k_encode_values<false>, g, b, 0, s, n, v, t.step_c, code, dec);
}

void launch_encode_sweep(const Tables &t, int channel, uint32_t lo, uint32_t hi, unsigned long long *bad,
                         hipStream_t s) {
    if (hi <= lo) return;
    const bool srgb = channel == 0 && t.srgb;
    const float *thr = channel == 0 ? t.thr_c : t.thr_a;
    const float *dec = channel == 0 ? t.dec_c : t.dec_a;
    if (srgb)
        hipLaunchKernelGGL(k_encode_sweep<true>, dim3(8192), dim3(256), 0, s, lo, hi, t.step_c, thr, dec, bad);
    else
        hipLaunchKernelGGL(k_encode_sweep<false>, dim3(8192), dim3(256), 0, s, lo, hi, t.step_c, thr, dec, bad);
}

void launch_debug_draw_list(const SceneDev &sc, const Tables &t, Frame &f, const uint32_t *moff, const uint32_t *ioff,
                            int4 *draw, uint32_t *mmask4, hipStream_t s) {
    if (!f.NB) return;
    dim3 g(blocks_for(f.NB, 256)), b(256);
    if (t.spp == 8)
        hipLaunchKernelGGL(k_debug_draw<8>, g, b, 0, s, f.NB, (const int2 *)f.binfo, sc.finfo, (const uint32_t *)f.boff,
                           (const uint2 *)f.bcnt, (const uint32_t *)f.items, (const uint32_t *)f.imask, moff, ioff, draw, mmask4);
    else if (t.spp == 16)
        hipLaunchKernelGGL(k_debug_draw<16>, g, b, 0, s, f.NB, (const int2 *)f.binfo, sc.finfo, (const uint32_t *)f.boff,
                           (const uint2 *)f.bcnt, (const uint32_t *)f.items, (const uint32_t *)f.imask, moff, ioff, draw, mmask4);
    else
        hipLaunchKernelGGL(k_debug_draw<32>, g, b, 0, s, f.NB, (const int2 *)f.binfo, sc.finfo, (const uint32_t *)f.boff,
                           (const uint2 *)f.bcnt, (const uint32_t *)f.items, (const uint32_t *)f.imask, moff, ioff, draw, mmask4);
}

void launch_count_reduce(const uint2 *bcnt, size_t n, unsigned long long *out, hipStream_t s) {
    hipLaunchKernelGGL(k_count_reduce, dim3(256), dim3(256), 0, s, bcnt, n, out);
}

void launch_debug_counts(const Frame &f, uint32_t *merged, uint32_t *items, hipStream_t s) {
    if (f.NB) hipLaunchKernelGGL(k_debug_counts, dim3(blocks_for(f.NB, 256)), dim3(256), 0, s, f.NB, (const uint2 *)f.bcnt, merged, items);
}

}  // namespace sl
