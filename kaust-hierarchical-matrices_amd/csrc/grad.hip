// Gradients of a loss L(Y), Y = H X, with respect to the low-rank factors
// (no reference counterpart; the backward of HMatrixVecMult):
//   dU_t = dY[rows_t] (V_t^T X[cols_t])^T      (m x r)
//   dV_t = X[cols_t] (U_t^T dY[rows_t])^T      (n x r)
// One kernel reads U and V once and writes dU and dV once, on the FP64 matrix
// cores; nothing but those four streams goes through memory.
#include <algorithm>

#include "hmx_device.h"
#include "hmx_internal.h"
#include "mfma.h"

namespace hmx {

constexpr int kGradCG = 2;       // 16-column groups per work item
constexpr int kGradWaves = 8;    // waves per workgroup
constexpr int kGradTallRows = 512;  // tiles of this dimension and more: a workgroup per item
constexpr int kGradLevels = 32;

// Destination of every level's gradients (kernel argument)
struct GradDst {
    double* dU[kGradLevels];
    double* dV[kGradLevels];
};

// one lane's 4 consecutive doubles
__device__ inline void ld4(const double* __restrict__ p, double (&o)[4]) {
    const double2 a = reinterpret_cast<const double2*>(p)[0], b = reinterpret_cast<const double2*>(p)[1];
    o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
}

// Up to 32 columns of one tile per item: Z^T = X^T V and G^T = dY^T U over
// the tile's rows, then dU = dY Z^T and dV = X G^T over the same rows.
//
// The transposed sums are formed (right-hand sides as the 16x16x4 product's
// rows, factor columns as its columns) because their result registers are
// then the next product's operand as they stand: lane (lg, lc), register v
// of Z^T holds (right-hand side 4v + lg, column lc), and step v of dU's
// product takes from lane (lg, lc) column lc at right-hand side 4v + lg. No
// Z in memory, no LDS for short tiles.  In the first product a lane takes 4
// consecutive rows of X and of V (whole 128-byte lines per column); both
// operands use the same row order.
//
// Items [0, nTall) are tiles of 512 rows and more: the workgroup's 8 waves
// take 16-row chunks in turn, their partial Z^T and G^T are folded in LDS in
// a fixed order, and every wave writes the gradient rows of its own chunks.
// The other items (largest first) take a wave each.  X and dY are the padded
// vectors (k right-hand sides, ld apart), read from the caches.
//
// Bound by HBM (32 bytes per factor entry pair) and by the matrix cores
// about equally at 32 right-hand sides.  N = 65536 2D, 32 right-hand sides
// (1.1 GB of factors, as much of gradients): 0.91 ms, 2.4 TB/s; a thread per
// gradient row, serial over columns and right-hand sides, with z in memory,
// took 89 ms.
template <int NB>
__global__ void __launch_bounds__(64 * kGradWaves) k_grad_tiles(const GradItem* __restrict__ items, int nTall, int nItems,
                                                                 GradDst dst, const double* __restrict__ X,
                                                                 const double* __restrict__ W, int64_t ld, int k,
                                                                 int accumulate) {
    using M = Mfma<double>;
    constexpr int CG = kGradCG, NW = kGradWaves, NQ = 4 * NB;
    __shared__ double red[NW][NQ][64];
    const int lane = threadIdx.x & 63, lg = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const bool tall = (int)blockIdx.x < nTall;
    const int id = tall ? (int)blockIdx.x : nTall + ((int)blockIdx.x - nTall) * NW + w;
    if (id >= nItems) return;  // whole waves, and only in blocks without barriers (not tall)
    const GradItem it = items[id];
    const int m = it.m, ncols = it.ncols;
    const int step = tall ? 16 * NW : 16, first = tall ? 16 * w : 0;
    const double *V = in_global<double>(it.V), *U = in_global<double>(it.U);
    const double* __restrict__ Xc = X + it.colStart;
    const double* __restrict__ Wr = W + it.rowStart;
    v4d zt[CG][NB], gt[CG][NB];
#pragma unroll
    for (int g = 0; g < CG; ++g)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            zt[g][nb] = v4d{0, 0, 0, 0};
            gt[g][nb] = v4d{0, 0, 0, 0};
        }
    for (int r0 = first; r0 < m; r0 += step) {
        const int r = r0 + 4 * lg;
        double xa[NB][4], wa[NB][4], vb[CG][4], ub[CG][4];
#pragma unroll
        for (int g = 0; g < CG; ++g) {
            if (16 * g + lc < ncols) {
                ld4(V + (size_t)(16 * g + lc) * m + r, vb[g]);
                ld4(U + (size_t)(16 * g + lc) * m + r, ub[g]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) vb[g][e] = ub[g][e] = 0.0;
            }
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (16 * nb + lc < k) {
                ld4(Xc + (size_t)(16 * nb + lc) * ld + r, xa[nb]);
                ld4(Wr + (size_t)(16 * nb + lc) * ld + r, wa[nb]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) xa[nb][e] = wa[nb][e] = 0.0;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int g = 0; g < CG; ++g)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    zt[g][nb] = M::op(xa[nb][e], vb[g][e], zt[g][nb]);
                    gt[g][nb] = M::op(wa[nb][e], ub[g][e], gt[g][nb]);
                }
    }
    if (tall) {
        // fold the waves' partial sums: wave q sums register q, q + 8, ... of
        // all waves in order, then every wave reads the sums
        auto fold = [&](v4d(&t)[NB]) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[w][4 * nb + v][lane] = t[nb][v];
            __syncthreads();
            for (int q = w; q < NQ; q += NW) {
                double s = red[0][q][lane];
#pragma unroll
                for (int p = 1; p < NW; ++p) s += red[p][q][lane];
                red[0][q][lane] = s;
            }
            __syncthreads();
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int v = 0; v < 4; ++v) t[nb][v] = red[0][4 * nb + v][lane];
            __syncthreads();
        };
#pragma unroll
        for (int g = 0; g < CG; ++g) {
            fold(zt[g]);
            fold(gt[g]);
        }
    }
    double* __restrict__ dU = dst.dU[it.level] + it.off;
    double* __restrict__ dV = dst.dV[it.level] + it.off;
    auto put = [&](double* __restrict__ d, int g, int r0, const v4d& o) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int a = 16 * g + M::out_row(lg, v);
            if (a < ncols) {
                double* p = d + (size_t)a * m + r0 + lc;
                *p = accumulate ? *p + o[v] : o[v];
            }
        }
    };
    for (int r0 = first; r0 < m; r0 += step) {
        double wb[NB][4], xb[NB][4];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int s = 16 * nb + 4 * t + lg;
                wb[nb][t] = s < k ? Wr[(size_t)s * ld + r0 + lc] : 0.0;
                xb[nb][t] = s < k ? Xc[(size_t)s * ld + r0 + lc] : 0.0;
            }
#pragma unroll
        for (int g = 0; g < CG; ++g) {
            v4d du = v4d{0, 0, 0, 0}, dv = v4d{0, 0, 0, 0};
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    du = M::op(zt[g][nb][t], wb[nb][t], du);
                    dv = M::op(gt[g][nb][t], xb[nb][t], dv);
                }
            put(dU, g, r0, du);
            put(dV, g, r0, dv);
        }
    }
}

// The work list of an H-matrix's tiles: tall tiles first, then by falling
// dimension.  The factors' places do not change while the H-matrix lives.
static void build_grad_plan(Context& c, const HMatrix& h, GradPlan& P) {
    HMX_CHECK(h.numLevels <= kGradLevels, HMX_EUNSUPPORTED, "factor gradients: too many levels");
    HMX_CHECK(h.b == 32 || h.b == 64, HMX_EUNSUPPORTED, "the factor-gradient kernel is built for bucketSize 32 or 64");
    std::vector<GradItem> items;
    for (int l = 1; l < h.numLevels; ++l) {  // level 1 holds the largest tiles
        const HLevel& lv = h.levels[l - 1];
        const auto& ti = h.structure->tileIndices[l - 1];
        for (int t = 0; t < lv.numTiles; ++t) {
            const int r = lv.h_ranks[t];
            const uint32_t u = compact16((uint32_t)ti[t]), v = compact16((uint32_t)ti[t] >> 1);
            for (int c0 = 0; c0 < r; c0 += 16 * kGradCG) {
                const int64_t off = (lv.h_offsets[t] + c0) * lv.m;
                items.push_back(GradItem{lv.U.p + off, lv.V.p + off, off, l - 1, lv.m,
                                         std::min(r - c0, 16 * kGradCG), (int32_t)(v * lv.m), (int32_t)(u * lv.m), 0});
            }
        }
        if (lv.m >= kGradTallRows) P.numTall = (int32_t)items.size();
    }
    P.numItems = (int32_t)items.size();
    P.items.alloc(std::max<size_t>(1, items.size()));
    if (!items.empty())
        HMX_HIP(hipMemcpyAsync(P.items.p, items.data(), items.size() * sizeof(GradItem), hipMemcpyHostToDevice, c.stream));
    P.npad = (int64_t)h.S * h.b;
    if (P.npad != (int64_t)h.n) {
        HMX_CHECK(h.leafOffsets.size() == (size_t)h.S + 1, HMX_ESTATE, "H-matrix without leaf offsets");
        const std::vector<int32_t> gm = padding_map(h, 0);
        P.gmap.alloc(gm.size());
        HMX_HIP(hipMemcpyAsync(P.gmap.p, gm.data(), gm.size() * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
        HMX_HIP(hipStreamSynchronize(c.stream));
    }
    HMX_HIP(hipStreamSynchronize(c.stream));
    P.built = true;
}

void hmatvec_grad_factors(Context& c, HMatrix& h, uint32_t k, const double* X, const double* dY,
                          double* const* dU, double* const* dV) {
    HMX_CHECK(k >= 1, HMX_EINVAL, "vectorWidth must be >= 1");
    HMX_CHECK(X && dY && dU && dV, HMX_EINVAL, "null pointer");
    GradDst dst{};
    bool any = false;
    for (int l = 0; l + 1 < h.numLevels; ++l) {
        if (h.levels[l].rankSum == 0) continue;
        HMX_CHECK(l < kGradLevels, HMX_EUNSUPPORTED, "factor gradients: too many levels");
        HMX_CHECK(dU[l] && dV[l], HMX_EINVAL, "null gradient buffer for a non-empty level");
        dst.dU[l] = dU[l];
        dst.dV[l] = dV[l];
        any = true;
    }
    if (!any) return;
    GradPlan& P = h.grad;
    if (!P.built) build_grad_plan(c, h, P);
    // The kernel reads the right-hand sides in the padded leaf space (zero on
    // padding rows, so the padding rows of dU and dV come out zero as the
    // factors' own are) with 16-byte loads: partial leaves are gathered, and
    // vectors that do not start on 16 bytes copied.
    const bool gather = P.npad != (int64_t)h.n;
    const bool copy = !gather && (((uintptr_t)X | (uintptr_t)dY) & 15);
    const int NB = mf_pass_blocks(k), NR = 16 * NB;
    if (gather || copy) {
        grow(P.Xp, (size_t)P.npad * NR);
        grow(P.Wp, (size_t)P.npad * NR);
    }
    for (uint32_t s0 = 0; s0 < k; s0 += NR) {
        const int kk = (int)std::min<uint32_t>(NR, k - s0);
        const double* Xs = X + (size_t)s0 * h.n;
        const double* Ws = dY + (size_t)s0 * h.n;
        if (gather) {
            gather_padded(c, P.npad, kk, P.gmap.p, Xs, h.n, P.Xp.p);
            gather_padded(c, P.npad, kk, P.gmap.p, Ws, h.n, P.Wp.p);
        } else if (copy) {
            const size_t bytes = (size_t)P.npad * kk * sizeof(double);
            HMX_HIP(hipMemcpyAsync(P.Xp.p, Xs, bytes, hipMemcpyDeviceToDevice, c.stream));
            HMX_HIP(hipMemcpyAsync(P.Wp.p, Ws, bytes, hipMemcpyDeviceToDevice, c.stream));
        }
        const bool own = gather || copy;
        const unsigned blocks = (unsigned)(P.numTall + (P.numItems - P.numTall + kGradWaves - 1) / kGradWaves);
        auto kern = NB == 1 ? k_grad_tiles<1> : NB == 2 ? k_grad_tiles<2> : NB == 3 ? k_grad_tiles<3> : k_grad_tiles<4>;
        kern<<<blocks, 64 * kGradWaves, 0, c.stream>>>(P.items.p, P.numTall, P.numItems, dst, own ? P.Xp.p : Xs,
                                                       own ? P.Wp.p : Ws, P.npad, kk, s0 > 0 ? 1 : 0);
        HMX_LAUNCHED();
    }
    HMX_HIP(hipStreamSynchronize(c.stream));
}

// overwrite one level's factors (device buffers in the level's layout)
void hmatrix_set_level(Context& c, HMatrix& h, int level, const double* U, const double* V) {
    HMX_CHECK(level >= 1 && level < h.numLevels, HMX_EINVAL, "level out of range");
    HLevel& lv = h.levels[level - 1];
    if (lv.U.n) {
        HMX_CHECK(U && V, HMX_EINVAL, "null factor buffer");
        HMX_HIP(hipMemcpyAsync(lv.U.p, U, lv.U.bytes(), hipMemcpyDeviceToDevice, c.stream));
        HMX_HIP(hipMemcpyAsync(lv.V.p, V, lv.V.bytes(), hipMemcpyDeviceToDevice, c.stream));
    }
    HMX_HIP(hipStreamSynchronize(c.stream));
    // converted copies used by the matrix-core paths, and the streaming
    // plans' dense near-field blocks, are stale now
    ++h.factorGen;
    h.mf64 = MfPlan();
    h.mf64T = MfPlan();
    h.mfMixed = MfPlan();
    h.plan = MatvecPlan();
    h.planT = MatvecPlan();
}

}  // namespace hmx
