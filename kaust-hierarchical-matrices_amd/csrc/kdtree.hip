// KD-tree construction, FULL_TREE division (src/kDTreeConstruction.cu:14-231).
//
// Per level: (1) segmented min/max over every dimension -> bounding boxes and
// split dimension (first maximal span, CUB ArgMax semantics); (2) stable
// ascending sort of each segment by the split coordinate; (3) each segment is
// split at a + ceil((e-a)/2).  Offsets depend only on n, so every level's
// tables are made on the host and uploaded once, and the levels run without
// a host wait between them.
//
//   * Each coordinate is sorted once (stable LSD radix sort of the 64-bit
//     keys) and replaced by its rank, equal values by equal ranks.  A level's
//     stable sort is then 2 to 4 radix passes over 32-bit ranks instead of 8
//     over 64-bit keys, and gives the same order, ties included.
//   * Segments of at most 2048 points finish all their levels in one
//     workgroup: the points stay in LDS, boxes by wave reductions, sorts by a
//     bitonic network on the unique (key, position) pair, which equals a
//     stable sort.
//
// N = 2^20 3D, leaves of 64: 2.3 ms with the copies to the host; a radix
// sort of the 64-bit keys per level, one launch and one wait per level also
// for the small segments, took 7.3 (2.8 of it in the serial digit offsets).
//
// Many clouds of the same dimension are built as one forest: their points
// side by side, every level's segments of every cloud sorted by the same
// launches, so a batch of clouds costs launches per level, not per cloud.
// Each segment is processed exactly as in a one-cloud build, so every tree
// is bitwise the tree its cloud gets alone.
#include <algorithm>
#include <cfloat>

#include "hmx_device.h"
#include "hmx_internal.h"

namespace hmx {

constexpr int kSmallSeg = 2048;    // points a workgroup finishes in LDS
constexpr int kSmallThreads = 512;
constexpr int kRadixChunk = 2048;  // points per workgroup of the large segments' kernels
constexpr int kWideScan = 32;      // chunks per segment from which the digit offsets take several workgroups

// A large segment of one level: its first position, its chunks, its box slot
struct KdSeg {
    int32_t start, c0, c1, pad;
    int64_t node;
};

// A segment that one workgroup finishes: positions [start, start + size),
// number seg of its cloud's level 'level', levels level .. L-1 still to split;
// 2^lgP points of LDS (sizes of its level are at most 2^lgP); p2l: cut at
// halves of 2^lgP (POWER_OF_TWO_ON_LEFT), else in halves
struct KdSmall {
    int32_t start, size, seg, level, L, lgP, p2l, pad;
    int64_t nodeBase;
};

// ---- large segments ------------------------------------------------------------
// points interleaved (x, y, z, 0), identity permutation, and zeros in the box
// slots (nbox values): no level fills those of the leaves and of segments a
// tree does not have
__global__ void __launch_bounds__(256) k_kd_init(int64_t n, uint32_t d, const double* __restrict__ p,
                                                 double4* __restrict__ P4, int32_t* __restrict__ perm, int64_t nbox,
                                                 double* __restrict__ bbmin, double* __restrict__ bbmax) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < nbox) bbmin[e] = bbmax[e] = 0.0;
    if (e >= n) return;
    perm[e] = (int32_t)e;
    if (!P4) return;
    const double x = p[e], y = d > 1 ? p[(size_t)n + e] : 0.0, z = d > 2 ? p[2 * (size_t)n + e] : 0.0;
    P4[e] = make_double4(x, y, z, 0.0);
}

// keys and values of nd coordinates, one after the other
__global__ void __launch_bounds__(256) k_kd_keys(int64_t n, int64_t tot, const double* __restrict__ p,
                                                 uint64_t* __restrict__ keys, int32_t* __restrict__ vals) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= tot) return;
    keys[e] = dkey(p[e]);
    vals[e] = (int32_t)(e % n);
}

// rank of every point in one sorted coordinate: the position of the first
// key equal to its own
__global__ void __launch_bounds__(256) k_kd_ranks(int64_t n, int64_t tot, const uint64_t* __restrict__ keys,
                                                  const int32_t* __restrict__ vals, uint32_t* __restrict__ rank) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= tot) return;
    const int64_t base = e / n * n;
    const uint64_t key = keys[e];
    int64_t r = e;
    if (e > base && keys[e - 1] == key) {  // a tie: binary search for its first
        int64_t lo = base, hi = e - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (keys[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        r = lo;
    }
    rank[base + vals[e]] = (uint32_t)(r - base);
}

// min/max of one chunk, all dims (chunks: {start, end, segment, -})
__global__ void __launch_bounds__(256) k_bbox_partial(uint32_t d, const double4* __restrict__ P4,
                                                      const int32_t* __restrict__ perm,
                                                      const int4* __restrict__ chunks, double* __restrict__ pmin,
                                                      double* __restrict__ pmax) {
    __shared__ double smin[4][3], smax[4][3];
    const int4 ch = chunks[blockIdx.x];
    double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    const int cnt = ch.y - ch.x;  // positions reach 2^31 - 1: only offsets are stepped
#pragma unroll 4
    for (int o = threadIdx.x; o < cnt; o += 256) {
        const double4 q = P4[perm[ch.x + o]];
        const double v[3] = {q.x, q.y, q.z};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            mn[j] = v[j] < mn[j] ? v[j] : mn[j];
            mx[j] = v[j] > mx[j] ? v[j] : mx[j];
        }
    }
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double a = __shfl_xor(mn[j], off, 64), b = __shfl_xor(mx[j], off, 64);
            mn[j] = a < mn[j] ? a : mn[j];
            mx[j] = b > mx[j] ? b : mx[j];
        }
        if ((threadIdx.x & 63) == 0) {
            smin[w][j] = mn[j];
            smax[w][j] = mx[j];
        }
    }
    __syncthreads();
    if (threadIdx.x < d) {
        const int j = threadIdx.x;
        double a = smin[0][j], b = smax[0][j];
        for (int q = 1; q < 4; ++q) {
            a = smin[q][j] < a ? smin[q][j] : a;
            b = smax[q][j] > b ? smax[q][j] : b;
        }
        pmin[(size_t)blockIdx.x * d + j] = a;
        pmax[(size_t)blockIdx.x * d + j] = b;
    }
}

// first dimension of maximal span (findSpan + ArgMax, src/kDTreeHelpers.cu:52-64)
__device__ inline int widest(uint32_t d, const double (&mn)[3], const double (&mx)[3]) {
    int dim = 0;
    double best = mx[0] - mn[0];
    for (uint32_t j = 1; j < d; ++j) {
        const double sp = mx[j] - mn[j];
        if (sp > best) { best = sp; dim = (int)j; }
    }
    return dim;
}

// one wave per segment: fold the chunk partials, write the segment's box and
// the split dimension
__global__ void __launch_bounds__(64) k_bbox_final(uint32_t d, const KdSeg* __restrict__ segs,
                                                   const double* __restrict__ pmin, const double* __restrict__ pmax,
                                                   double* __restrict__ bbmin, double* __restrict__ bbmax,
                                                   int32_t* __restrict__ splitDim) {
    const KdSeg sg = segs[blockIdx.x];
    double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (int c = sg.c0 + threadIdx.x; c < sg.c1; c += 64)
        for (uint32_t j = 0; j < d; ++j) {
            const double a = pmin[(size_t)c * d + j], b = pmax[(size_t)c * d + j];
            if (a < mn[j]) mn[j] = a;
            if (b > mx[j]) mx[j] = b;
        }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double a = __shfl_xor(mn[j], off, 64), b = __shfl_xor(mx[j], off, 64);
            if (a < mn[j]) mn[j] = a;
            if (b > mx[j]) mx[j] = b;
        }
    if (threadIdx.x == 0) {
        for (uint32_t j = 0; j < d; ++j) {
            bbmin[sg.node * d + j] = mn[j];
            bbmax[sg.node * d + j] = mx[j];
        }
        splitDim[blockIdx.x] = widest(d, mn, mx);
    }
}

// Digit counts of every chunk; GATHER: the keys are the ranks of the
// segment's split coordinate, gathered through the permutation and kept
template <class KT, bool GATHER>
__global__ void __launch_bounds__(256) k_radix_hist(KT* __restrict__ keys, const int4* __restrict__ chunks, int shift,
                                                    int mask, int32_t* __restrict__ hist,
                                                    const uint32_t* __restrict__ rank, int64_t n,
                                                    const int32_t* __restrict__ perm,
                                                    const int32_t* __restrict__ splitDim) {
    __shared__ int32_t cnt[256];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int4 ch = chunks[blockIdx.x];
    const uint32_t* rk = GATHER ? rank + (size_t)splitDim[ch.z] * n : nullptr;
    const int size = ch.y - ch.x;
#pragma unroll 4
    for (int o = threadIdx.x; o < size; o += 256) {
        const int i = ch.x + o;
        KT k;
        if constexpr (GATHER) {
            k = rk[perm[i]];
            keys[i] = k;
        } else {
            k = keys[i];
        }
        atomicAdd(&cnt[(int)(k >> shift) & mask], 1);
    }
    __syncthreads();
    hist[(size_t)blockIdx.x * 256 + threadIdx.x] = cnt[threadIdx.x];
}

// Offsets of every chunk's digits inside their digit, and the segment's digit
// totals.  Segments of few chunks: one workgroup each, thread = digit.
__global__ void __launch_bounds__(256) k_radix_offsets(const int32_t* __restrict__ hist, const KdSeg* __restrict__ segs,
                                                       int32_t* __restrict__ choff, int32_t* __restrict__ total) {
    const KdSeg sg = segs[blockIdx.x];
    const int d = threadIdx.x;
    int run = 0;
#pragma unroll 4
    for (int c = sg.c0; c < sg.c1; ++c) {
        const int v = hist[(size_t)c * 256 + d];
        choff[(size_t)c * 256 + d] = run;
        run += v;
    }
    total[(size_t)blockIdx.x * 256 + d] = run;
}

// The same for long segments: 16 workgroups per segment, 16 digits each, 16
// runs of chunks per digit (one workgroup, serial over 512 chunks twice, took
// 130 us at the first level of 2^20 points)
__global__ void __launch_bounds__(256) k_radix_offsets_wide(const int32_t* __restrict__ hist,
                                                            const KdSeg* __restrict__ segs,
                                                            int32_t* __restrict__ choff, int32_t* __restrict__ total) {
    __shared__ int32_t part[16][16];
    const KdSeg sg = segs[blockIdx.y];
    const int dd = threadIdx.x & 15, q = threadIdx.x >> 4, d = blockIdx.x * 16 + dd;
    const int C = sg.c1 - sg.c0, per = (C + 15) / 16;
    const int a = sg.c0 + min(C, q * per), e = sg.c0 + min(C, (q + 1) * per);
    int sum = 0;
#pragma unroll 8
    for (int c = a; c < e; ++c) sum += hist[(size_t)c * 256 + d];
    part[q][dd] = sum;
    __syncthreads();
    int run = 0, all = 0;
    for (int r = 0; r < 16; ++r) {
        if (r == q) run = all;
        all += part[r][dd];
    }
#pragma unroll 8
    for (int c = a; c < e; ++c) {
        const int v = hist[(size_t)c * 256 + d];
        choff[(size_t)c * 256 + d] = run;
        run += v;
    }
    if (q == 0) total[(size_t)blockIdx.y * 256 + d] = all;
}

// stable scatter: 4 waves, wave w owns elements [w*512, w*512+512) of the chunk
template <class KT>
__global__ void __launch_bounds__(256) k_radix_scatter(const KT* __restrict__ keys, const int32_t* __restrict__ vin,
                                                       const int4* __restrict__ chunks, const KdSeg* __restrict__ segs,
                                                       int shift, int mask, const int32_t* __restrict__ choff,
                                                       const int32_t* __restrict__ total, KT* __restrict__ kout,
                                                       int32_t* __restrict__ vout) {
    __shared__ int32_t cnt[4][256];
    __shared__ int32_t wsum[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * 256; i += 256) (&cnt[0][0])[i] = 0;
    const int4 ch = chunks[blockIdx.x];
    // the digits' first positions: an exclusive sum over the segment's totals
    const int tot = total[(size_t)ch.z * 256 + threadIdx.x];
    int inc = tot;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(inc, off, 64);
        if (lane >= off) inc += v;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    constexpr int per = kRadixChunk / 4, RD = per / 64;
    int32_t rk[RD], dg[RD], val[RD];
    KT key[RD];
    const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    const int size = ch.y - ch.x;
#pragma unroll
    for (int r = 0; r < RD; ++r) {
        const int o = w * per + r * 64 + lane;
        const bool valid = o < size;
        key[r] = valid ? keys[ch.x + o] : (KT)0;
        val[r] = valid ? vin[ch.x + o] : 0;
    }
#pragma unroll
    for (int r = 0; r < RD; ++r) {
        const bool valid = w * per + r * 64 + lane < size;
        const int d = (int)(key[r] >> shift) & mask;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool on = (d >> bit) & 1;
            const uint64_t bal = __ballot(valid && on);
            peers &= on ? bal : ~bal;
        }
        const int before = valid ? cnt[w][d] : 0;
        const int rl = __popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (valid && rl == 0) cnt[w][d] = before + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rk[r] = before + rl;
        dg[r] = valid ? d : -1;
    }
    __syncthreads();
    {
        const int d = threadIdx.x;
        int run = segs[ch.z].start + inc - tot + choff[(size_t)blockIdx.x * 256 + d];
        for (int q = 0; q < w; ++q) run += wsum[q];
        for (int q = 0; q < 4; ++q) {
            const int v = cnt[q][d];
            cnt[q][d] = run;
            run += v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RD; ++r) {
        if (dg[r] < 0) continue;
        const int dst = cnt[w][dg[r]] + rk[r];
        kout[dst] = key[r];
        vout[dst] = val[r];
    }
}

// ---- small segments: all remaining levels in LDS -------------------------------
// The points of sub-segment q of a level sit in slot q, 2^lg places of which
// the first cnt(q) are used; a level's boxes and split dimensions by wave
// reductions, its sorts by one bitonic network over all slots, and the two
// halves of a sorted slot move to the two slots of half its size.
template <int D>
__global__ void __launch_bounds__(kSmallThreads) k_kd_small(int64_t n, const double* __restrict__ p,
                                                            int32_t* __restrict__ perm,
                                                            const KdSmall* __restrict__ segs,
                                                            double* __restrict__ bbmin, double* __restrict__ bbmax) {
    constexpr int NT = kSmallThreads, NW = NT / 64, E = kSmallSeg / NT;
    __shared__ double x[D][kSmallSeg];
    __shared__ uint64_t key[kSmallSeg];
    __shared__ uint16_t pos[kSmallSeg];
    __shared__ int32_t idx[kSmallSeg];
    __shared__ uint8_t dim[kSmallSeg];
    __shared__ double wmin[NW][3], wmax[NW][3];
    const KdSmall sg = segs[blockIdx.x];
    const int P = 1 << sg.lgP, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    for (int i = tid; i < sg.size; i += NT) {
        const int32_t v = perm[sg.start + i];
        idx[i] = v;
#pragma unroll
        for (int j = 0; j < D; ++j) x[j][i] = p[(size_t)j * n + v];
    }
    __syncthreads();
    // points and first point (of the segment) of sub-segment q, t levels down
    auto part = [&](int q, int t, int& off) {
        if (sg.p2l) {
            const int s = P >> t;
            off = q * s;
            return min(s, max(0, sg.size - off));
        }
        int c = sg.size;
        off = 0;
        for (int b = t - 1; b >= 0; --b) {
            const int h = (c + 1) >> 1;
            if ((q >> b) & 1) {
                off += h;
                c -= h;
            } else {
                c = h;
            }
        }
        return c;
    };
    for (int level = sg.level; level < sg.L; ++level) {
        const int t = level - sg.level, lg = sg.lgP - t, nsub = 1 << t;
        // boxes: NW / nsub waves per sub-segment, or sub-segments in turn
        const int wps = nsub < NW ? NW / nsub : 1;
        for (int q0 = 0; q0 < nsub; q0 += NW / wps) {
            const int q = q0 + w / wps, r = w % wps;
            double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
            int off = 0, c = 0;
            if (q < nsub) {
                c = part(q, t, off);
                for (int o = r * 64 + lane; o < c; o += 64 * wps)
#pragma unroll
                    for (int j = 0; j < D; ++j) {
                        const double v = x[j][(q << lg) + o];
                        mn[j] = v < mn[j] ? v : mn[j];
                        mx[j] = v > mx[j] ? v : mx[j];
                    }
            }
#pragma unroll
            for (int j = 0; j < D; ++j)
#pragma unroll
                for (int s = 32; s > 0; s >>= 1) {
                    const double a = __shfl_xor(mn[j], s, 64), b = __shfl_xor(mx[j], s, 64);
                    mn[j] = a < mn[j] ? a : mn[j];
                    mx[j] = b > mx[j] ? b : mx[j];
                }
            if (wps > 1) {
                if (lane < D) {
                    wmin[w][lane] = lane == 0 ? mn[0] : lane == 1 ? mn[1] : mn[2];
                    wmax[w][lane] = lane == 0 ? mx[0] : lane == 1 ? mx[1] : mx[2];
                }
                __syncthreads();
                if (r == 0)
                    for (int v = 1; v < wps; ++v)
#pragma unroll
                        for (int j = 0; j < D; ++j) {
                            const double a = wmin[w + v][j], b = wmax[w + v][j];
                            mn[j] = a < mn[j] ? a : mn[j];
                            mx[j] = b > mx[j] ? b : mx[j];
                        }
            }
            // POWER_OF_TWO_ON_LEFT has no empty segments: nothing to write for one
            if (q < nsub && r == 0 && lane == 0 && (c > 0 || !sg.p2l)) {
                const int64_t o = (sg.nodeBase + ((int64_t)1 << level) - 1 + ((int64_t)sg.seg << t) + q) * D;
#pragma unroll
                for (int j = 0; j < D; ++j) {
                    bbmin[o + j] = mn[j];
                    bbmax[o + j] = mx[j];
                }
                dim[q] = (uint8_t)widest(D, mn, mx);
            }
        }
        __syncthreads();
        for (int i = tid; i < P; i += NT) {
            const int q = i >> lg, o = i & ((1 << lg) - 1);
            int off;
            const bool used = o < part(q, t, off);
            key[i] = used ? dkey(x[dim[q]][i]) : ~0ull;
            pos[i] = (uint16_t)o;
        }
        __syncthreads();
        for (int k = 2; k <= 1 << lg; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int e = tid; e < P / 2; e += NT) {
                    const int i = ((e & ~(j - 1)) << 1) | (e & (j - 1)), l = i | j;
                    const uint64_t ka = key[i], kb = key[l];
                    const uint16_t pa = pos[i], pb = pos[l];
                    const bool gt = ka > kb || (ka == kb && pa > pb);
                    const bool asc = ((i & ((1 << lg) - 1)) & k) == 0;
                    if (gt == asc) {
                        key[i] = kb; key[l] = ka;
                        pos[i] = pb; pos[l] = pa;
                    }
                }
                __syncthreads();
            }
        // every point to its place in the next level's slots, or to the permutation
        int32_t mv[E], to[E];
        double mx[E][D];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const int i = tid + u * NT;
            to[u] = -1;
            if (i >= P) continue;
            const int q = i >> lg, o = i & ((1 << lg) - 1);
            int off;
            const int c = part(q, t, off);
            if (o >= c) continue;
            const int src = (q << lg) + pos[i];
            mv[u] = idx[src];
            if (level + 1 == sg.L) {
                perm[sg.start + off + o] = mv[u];
                continue;
            }
#pragma unroll
            for (int j = 0; j < D; ++j) mx[u][j] = x[j][src];
            const int h = sg.p2l ? 1 << (lg - 1) : (c + 1) >> 1;
            to[u] = o < h ? (q << lg) + o : (q << lg) + (1 << (lg - 1)) + o - h;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < E; ++u)
            if (to[u] >= 0) {
                idx[to[u]] = mv[u];
#pragma unroll
                for (int j = 0; j < D; ++j) x[j][to[u]] = mx[u][j];
            }
        __syncthreads();
    }
}

// positions of a level's chunks from one permutation buffer to the other
__global__ void __launch_bounds__(256) k_copy_segments(const int4* __restrict__ chunks, const int32_t* __restrict__ src,
                                                       int32_t* __restrict__ dst) {
    const int4 ch = chunks[blockIdx.x];
    for (int o = threadIdx.x; o < ch.y - ch.x; o += 256) dst[ch.x + o] = src[ch.x + o];
}

// the forest's points side by side: Pc[j * ntot + base_k + i] = p_k[j * n_k + i]
struct KdSrc {
    int64_t base;
    const double* p;
    uint32_t n;
};

__global__ void __launch_bounds__(256) k_forest_gather(int64_t ntot, uint32_t d, const KdSrc* __restrict__ src, int ns,
                                                       double* __restrict__ Pc) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= ntot) return;
    int lo = 0, hi = ns - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (src[mid].base <= e) lo = mid;
        else hi = mid - 1;
    }
    const KdSrc q = src[lo];
    const int64_t i = e - q.base;
    for (uint32_t j = 0; j < d; ++j) Pc[(size_t)j * ntot + e] = q.p[(size_t)j * q.n + i];
}

// forest positions back to each cloud's own point numbers
__global__ void __launch_bounds__(256) k_forest_localize(int64_t ntot, const KdSrc* __restrict__ src, int ns,
                                                         int32_t* __restrict__ perm) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= ntot) return;
    int lo = 0, hi = ns - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (src[mid].base <= e) lo = mid;
        else hi = mid - 1;
    }
    perm[e] -= (int32_t)src[lo].base;
}

// One cloud of a forest: its cuts at the current level, in its own positions
struct KdJob {
    KDTree* t;
    const double* p;
    int64_t base = 0;      // first position in the forest
    int64_t nodeBase = 0;  // first box slot in the forest's box arrays
    uint32_t L = 0, size = 0;
    bool p2l = false, small = false;  // small: its segments are with k_kd_small
    std::vector<int32_t> off;
};

// cuts of a cloud at a level: FULL_TREE / DIVIDE_IN_HALF split every segment
// at a + ceil((e-a)/2) (fillOffsetsSort, src/kDTreeHelpers.cu:81-93);
// POWER_OF_TWO_ON_LEFT cuts at multiples of a power-of-two size that starts
// at upperPowerOfTwo(n) and halves while it exceeds b (fillOffsets,
// src/kDTreeHelpers.cu:29-43)
static void p2l_cuts(uint32_t n, uint32_t lsize, std::vector<int32_t>& off) {
    const uint32_t ns = (n + lsize - 1) / lsize;
    off.assign(ns + 1, 0);
    for (uint32_t q = 0; q < ns; ++q) off[q] = (int32_t)(q * lsize);
    off[ns] = (int32_t)n;
}

// cuts of the next level: every segment in halves, the left one the longer
static std::vector<int32_t> halved(const std::vector<int32_t>& off) {
    const size_t ns = off.size() - 1;
    std::vector<int32_t> out(2 * ns + 1);
    for (size_t s = 0; s < ns; ++s) {
        out[2 * s] = off[s];
        out[2 * s + 1] = (off[s + 1] - off[s] + 1) / 2 + off[s];
    }
    out[2 * ns] = off[ns];
    return out;
}

static void kd_forest(Context& c, uint32_t d, std::vector<KdJob>& jobs) {
    const int nj = (int)jobs.size();
    int64_t ntot = 0, nodes = 0;
    uint32_t maxL = 0;
    for (KdJob& J : jobs) {
        KDTree& t = *J.t;
        HMX_CHECK(t.d == d, HMX_EINVAL, "a forest needs one dimension");
        HMX_CHECK(t.d >= 1 && t.d <= 3, HMX_EINVAL, "dimensionOfInputPoints must be 1, 2 or 3");
        HMX_CHECK(t.b >= 1, HMX_EINVAL, "bucketSize must be >= 1");
        HMX_CHECK(t.n >= 1, HMX_EINVAL, "numberOfInputPoints must be >= 1");
        HMX_CHECK(J.p != nullptr, HMX_EINVAL, "null points");
        J.p2l = t.divMethod == HMX_POWER_OF_TWO_ON_LEFT;
        if (J.p2l) {
            J.size = upper_pow2(t.n);
            J.L = 0;
            while (J.size > t.b) { J.size >>= 1; ++J.L; }
            t.numSegments = (t.n + J.size - 1) / J.size;
        } else {
            J.L = kd_num_levels(t.n, t.b);
            t.numSegments = 1u << J.L;
        }
        t.numLevels = J.L;
        J.base = ntot;
        J.nodeBase = nodes;
        J.off = {0, (int32_t)t.n};
        ntot += t.n;
        nodes += ((int64_t)2 << J.L) - 1;
        maxL = std::max(maxL, J.L);
    }
    HMX_CHECK(ntot < ((int64_t)1 << 31), HMX_EINVAL, "a forest holds fewer than 2^31 points");
    // the points: one cloud is read where it lies; several are gathered side by side
    std::vector<KdSrc> hsrc(nj);
    for (int k = 0; k < nj; ++k) hsrc[k] = KdSrc{jobs[k].base, jobs[k].p, jobs[k].t->n};
    DBuf<KdSrc> dsrc(nj);
    HMX_HIP(hipMemcpyAsync(dsrc.p, hsrc.data(), nj * sizeof(KdSrc), hipMemcpyHostToDevice, c.stream));
    DBuf<double> Pc;
    const double* P = jobs[0].p;
    if (nj > 1) {
        Pc.alloc((size_t)ntot * d);
        k_forest_gather<<<(unsigned)((ntot + 255) / 256), 256, 0, c.stream>>>(ntot, d, dsrc.p, nj, Pc.p);
        HMX_LAUNCHED();
        P = Pc.p;
    }
    auto permF = std::make_shared<DBuf<int32_t>>((size_t)ntot);
    auto bbminF = std::make_shared<DBuf<double>>((size_t)nodes * d);
    auto bbmaxF = std::make_shared<DBuf<double>>((size_t)nodes * d);
    int32_t* perm = permF->p;

    // ---- the tables of all levels: the large segments of a level and their
    // chunks, and the segments that become small
    struct Level {
        size_t seg0, chunk0;
        int nseg, nchunk, maxChunks;
    };
    std::vector<Level> levels;
    std::vector<KdSeg> segs;
    std::vector<int4> chunks;
    std::vector<KdSmall> small;
    auto add_chunks = [&](Level& lv, int64_t start, int64_t end, int64_t node) {
        KdSeg sg{(int32_t)start, lv.nchunk, 0, 0, node};
        for (int64_t a = start; a < end; a += kRadixChunk, ++lv.nchunk)
            chunks.push_back(make_int4((int)a, (int)std::min<int64_t>(a + kRadixChunk, end), lv.nseg, 0));
        sg.c1 = lv.nchunk;
        lv.maxChunks = std::max(lv.maxChunks, sg.c1 - sg.c0);
        segs.push_back(sg);
        ++lv.nseg;
    };
    for (uint32_t level = 0; level < maxL; ++level) {
        Level lv{segs.size(), chunks.size(), 0, 0, 0};
        for (KdJob& J : jobs) {
            if (level >= J.L || J.small) continue;
            const uint32_t lsize = J.p2l ? J.size << (J.L - level) : (J.t->n + (1u << level) - 1) >> level;
            if (J.p2l) p2l_cuts(J.t->n, lsize, J.off);
            J.small = lsize <= (uint32_t)kSmallSeg;  // no segment of this level is longer
            int lgP = 0;
            while ((1u << lgP) < lsize) ++lgP;
            for (size_t s = 0; s + 1 < J.off.size(); ++s) {
                const int64_t a = J.base + J.off[s], e = J.base + J.off[s + 1];
                if (J.small)
                    small.push_back(KdSmall{(int32_t)a, (int32_t)(e - a), (int32_t)s, (int32_t)level, (int32_t)J.L, lgP,
                                            J.p2l ? 1 : 0, 0, J.nodeBase});
                else
                    add_chunks(lv, a, e, J.nodeBase + ((int64_t)1 << level) - 1 + (int64_t)s);
            }
        }
        if (lv.nseg) levels.push_back(lv);
        // ---- next level's cuts
        for (KdJob& J : jobs)
            if (level < J.L && !J.p2l) J.off = halved(J.off);
    }
    // a presort's segments: nd coordinates at once (32-bit positions)
    const int nd = ntot * d < ((int64_t)1 << 31) ? (int)d : 1;
    Level pre{segs.size(), chunks.size(), 0, 0, 0};
    const bool large = !levels.empty();
    if (large)
        for (int j = 0; j < nd; ++j) add_chunks(pre, j * ntot, (j + 1) * ntot, 0);
    DBuf<KdSeg> d_segs(std::max<size_t>(1, segs.size()));
    DBuf<int4> d_chunks(std::max<size_t>(1, chunks.size()));
    DBuf<KdSmall> d_small(std::max<size_t>(1, small.size()));
    if (large) {
        HMX_HIP(hipMemcpyAsync(d_segs.p, segs.data(), segs.size() * sizeof(KdSeg), hipMemcpyHostToDevice, c.stream));
        HMX_HIP(hipMemcpyAsync(d_chunks.p, chunks.data(), chunks.size() * sizeof(int4), hipMemcpyHostToDevice, c.stream));
    }
    if (!small.empty())
        HMX_HIP(hipMemcpyAsync(d_small.p, small.data(), small.size() * sizeof(KdSmall), hipMemcpyHostToDevice, c.stream));

    DBuf<double4> P4;
    if (large) P4.alloc((size_t)ntot);
    const int64_t nbox = nodes * d;
    k_kd_init<<<(unsigned)((std::max(ntot, nbox) + 255) / 256), 256, 0, c.stream>>>(ntot, d, P, P4.p, perm, nbox,
                                                                                    bbminF->p, bbmaxF->p);
    HMX_LAUNCHED();
    if (large) {
        int mostSegs = pre.nseg, mostChunks = pre.nchunk;
        for (const Level& lv : levels) {
            mostSegs = std::max(mostSegs, lv.nseg);
            mostChunks = std::max(mostChunks, lv.nchunk);
        }
        DBuf<int32_t> hist((size_t)mostChunks * 256), choff((size_t)mostChunks * 256), total((size_t)mostSegs * 256);
        auto offsets = [&](const Level& lv) {
            const KdSeg* sg = d_segs.p + lv.seg0;
            if (lv.maxChunks >= kWideScan)
                k_radix_offsets_wide<<<dim3(16, (unsigned)lv.nseg), 256, 0, c.stream>>>(hist.p, sg, choff.p, total.p);
            else
                k_radix_offsets<<<(unsigned)lv.nseg, 256, 0, c.stream>>>(hist.p, sg, choff.p, total.p);
            HMX_LAUNCHED();
        };
        // ---- ranks of every coordinate
        DBuf<uint32_t> rank((size_t)ntot * d);
        {
            const int64_t tot = ntot * nd;
            DBuf<uint64_t> ka((size_t)tot), kb((size_t)tot);
            DBuf<int32_t> va((size_t)tot), vb((size_t)tot);
            const unsigned grid = (unsigned)((tot + 255) / 256);
            for (uint32_t j = 0; j < d; j += (uint32_t)nd) {
                k_kd_keys<<<grid, 256, 0, c.stream>>>(ntot, tot, P + (size_t)j * ntot, ka.p, va.p);
                HMX_LAUNCHED();
                uint64_t *kin = ka.p, *kout = kb.p;
                int32_t *vin = va.p, *vout = vb.p;
                for (int shift = 0; shift < 64; shift += 8) {
                    k_radix_hist<uint64_t, false><<<(unsigned)pre.nchunk, 256, 0, c.stream>>>(
                        kin, d_chunks.p + pre.chunk0, shift, 255, hist.p, nullptr, 0, nullptr, nullptr);
                    HMX_LAUNCHED();
                    offsets(pre);
                    k_radix_scatter<uint64_t><<<(unsigned)pre.nchunk, 256, 0, c.stream>>>(
                        kin, vin, d_chunks.p + pre.chunk0, d_segs.p + pre.seg0, shift, 255, choff.p, total.p, kout, vout);
                    HMX_LAUNCHED();
                    std::swap(kin, kout);
                    std::swap(vin, vout);
                }
                k_kd_ranks<<<grid, 256, 0, c.stream>>>(ntot, tot, kin, vin, rank.p + (size_t)j * ntot);
                HMX_LAUNCHED();
            }
        }
        // ---- the levels
        int bits = 1;
        while (bits < 31 && ((int64_t)1 << bits) < ntot) ++bits;
        const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes, mask = (1 << width) - 1;
        DBuf<uint32_t> ka((size_t)ntot), kb((size_t)ntot);
        DBuf<int32_t> permB((size_t)ntot), splitDim((size_t)mostSegs);
        DBuf<double> pmin((size_t)mostChunks * d), pmax((size_t)mostChunks * d);
        for (const Level& lv : levels) {
            const KdSeg* sg = d_segs.p + lv.seg0;
            const int4* ch = d_chunks.p + lv.chunk0;
            const unsigned nch = (unsigned)lv.nchunk;
            k_bbox_partial<<<nch, 256, 0, c.stream>>>(d, P4.p, perm, ch, pmin.p, pmax.p);
            HMX_LAUNCHED();
            k_bbox_final<<<(unsigned)lv.nseg, 64, 0, c.stream>>>(d, sg, pmin.p, pmax.p, bbminF->p, bbmaxF->p, splitDim.p);
            HMX_LAUNCHED();
            uint32_t *kin = ka.p, *kout = kb.p;
            int32_t *vin = perm, *vout = permB.p;
            for (int pass = 0; pass < passes; ++pass) {
                const int shift = pass * width;
                if (pass == 0)
                    k_radix_hist<uint32_t, true><<<nch, 256, 0, c.stream>>>(kin, ch, shift, mask, hist.p, rank.p, ntot, vin,
                                                                            splitDim.p);
                else
                    k_radix_hist<uint32_t, false><<<nch, 256, 0, c.stream>>>(kin, ch, shift, mask, hist.p, nullptr, 0,
                                                                             nullptr, nullptr);
                HMX_LAUNCHED();
                offsets(lv);
                k_radix_scatter<uint32_t><<<nch, 256, 0, c.stream>>>(kin, vin, ch, sg, shift, mask, choff.p, total.p, kout,
                                                                     vout);
                HMX_LAUNCHED();
                std::swap(kin, kout);
                std::swap(vin, vout);
            }
            if (vin != perm) {  // odd number of passes: the level's positions back
                k_copy_segments<<<nch, 256, 0, c.stream>>>(ch, vin, perm);
                HMX_LAUNCHED();
            }
        }
    }
    if (!small.empty()) {
        auto k = d == 1 ? k_kd_small<1> : d == 2 ? k_kd_small<2> : k_kd_small<3>;
        k<<<(unsigned)small.size(), kSmallThreads, 0, c.stream>>>(ntot, P, perm, d_small.p, bbminF->p, bbmaxF->p);
        HMX_LAUNCHED();
    }
    if (nj > 1) {
        k_forest_localize<<<(unsigned)((ntot + 255) / 256), 256, 0, c.stream>>>(ntot, dsrc.p, nj, perm);
        HMX_LAUNCHED();
    }
    // leaf offsets of every tree in one block; boxes copied to the host once
    std::vector<int32_t> allOff;
    std::vector<int64_t> offBase(nj);
    for (int k = 0; k < nj; ++k) {
        KdJob& J = jobs[k];
        if (J.p2l) p2l_cuts(J.t->n, J.size, J.off);
        offBase[k] = (int64_t)allOff.size();
        allOff.insert(allOff.end(), J.off.begin(), J.off.end());
    }
    auto offF = std::make_shared<DBuf<int32_t>>(allOff.size());
    HMX_HIP(hipMemcpyAsync(offF->p, allOff.data(), allOff.size() * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
    std::vector<double> hmin((size_t)nodes * d), hmax((size_t)nodes * d);
    HMX_HIP(hipMemcpyAsync(hmin.data(), bbminF->p, hmin.size() * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    HMX_HIP(hipMemcpyAsync(hmax.data(), bbmaxF->p, hmax.size() * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    HMX_HIP(hipStreamSynchronize(c.stream));
    for (int k = 0; k < nj; ++k) {
        KdJob& J = jobs[k];
        KDTree& t = *J.t;
        const size_t nbox = ((size_t)2 << J.L) - 1;
        t.perm.view(permF, (size_t)J.base, t.n);
        t.offsets.view(offF, (size_t)offBase[k], J.off.size());
        t.bbmin.view(bbminF, (size_t)J.nodeBase * d, nbox * d);
        t.bbmax.view(bbmaxF, (size_t)J.nodeBase * d, nbox * d);
        t.h_offsets = J.off;
        t.h_bbmin.assign(hmin.begin() + J.nodeBase * d, hmin.begin() + (J.nodeBase + (int64_t)nbox) * d);
        t.h_bbmax.assign(hmax.begin() + J.nodeBase * d, hmax.begin() + (J.nodeBase + (int64_t)nbox) * d);
    }
}

void build_kdtree(Context& c, KDTree& t, const double* d_points) {
    HMX_CHECK(t.d >= 1 && t.d <= 3, HMX_EINVAL, "dimensionOfInputPoints must be 1, 2 or 3");
    std::vector<KdJob> jobs(1);
    jobs[0].t = &t;
    jobs[0].p = d_points;
    kd_forest(c, t.d, jobs);
}

// Trees of many clouds: one forest per point dimension
void build_kdtree_batch(Context& c, const std::vector<KDTree*>& ts, const std::vector<const double*>& pts) {
    HMX_CHECK(ts.size() == pts.size() && !ts.empty(), HMX_EINVAL, "batch arrays of different lengths");
    for (uint32_t d = 1; d <= 3; ++d) {
        std::vector<KdJob> jobs;
        for (size_t k = 0; k < ts.size(); ++k) {
            HMX_CHECK(ts[k]->d >= 1 && ts[k]->d <= 3, HMX_EINVAL, "dimensionOfInputPoints must be 1, 2 or 3");
            if (ts[k]->d != d) continue;
            jobs.emplace_back();
            jobs.back().t = ts[k];
            jobs.back().p = pts[k];
        }
        if (!jobs.empty()) kd_forest(c, d, jobs);
    }
}

}  // namespace hmx
