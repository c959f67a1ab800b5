// factor_tile.hip -- the per-column factorisation of the DEnKF and EnOI
// analyses, the per-obstype diagnostics and the adjoint's inverse, one
// wavefront per matrix, on 16 x 16 FP64 matrix-core tiles (tile_matrix.h).
//
// The work item of factor_tile_kernel is M = I + G0 of a stride-grid node, G0
// its full Gram matrix:
//   DEnKF  T = (I + M^-1) / 2 (first m_d rows), relaxed to the prior and cast
//          to FP32 (transforms.c:814-842);
//   w      = M^-1 S^T s;
//   dfs    = tr(M^-1 G0) = m - tr(M^-1)   (as M^-1 G0 = I - M^-1),
//   srf    = sqrt(tr(G0) / (float) dfs) - 1.
// factor_trace_kernel's is M_t = I + G_t of one (node, obstype) for the
// per-type diagnostics (calc/transforms.c:843-879), which need only
// tr(M_t^-1) and tr(G_t).
//
// M^-1 = V^T V from the block Cholesky factorisation, tr(M^-1) = |V|^2.  For
// m = 96 that is 50 tile products for the factor, 56 for V and 56 more for
// the whole inverse, of four MFMA instructions each, and six 16 x 16 factors.
// Bound: the FP64 matrix cores (64 cycles an instruction, 27k cycles a trace)
// and, beside them, the chain of 96 dependent pivots; two wavefronts share a
// SIMD up to m = 96, so that one's pivots run beside the other's products.
// The padding
// (rows m ..) is an identity block, which the elimination leaves intact.
//
// Measured against the kernels before it, which kept a matrix in 4 x 4 to 10 x
// 10 blocks on 192 lanes and swept one pivot per workgroup barrier: 51x1500x
// 1800 tile (300,000 nodes and 1.2M (node, type) matrices, m = 96) FP64 calc
// 468 -> 412 ms, mixed 269 -> 201 ms; 540x801 cells, factor alone 29 -> 6.7
// ms; 96 + 48 members on 8,000 nodes 10.2 -> 5.4 ms; m = 130, EnOI 2.9 -> 1.4
// ms.  For MT >= 7 one wavefront per SIMD holds its tiles in 512 registers;
// some MT spill (tile_waves).  Counters on the tile, the kernels alone: matrix
// cores busy 51% of a trace launch and 30% of a node launch, VALU issue 38%
// and 27%.
#include "enkfg_internal.h"
#include "gram_layout.h"
#include "tile_matrix.h"

namespace enkfg {

namespace {

template <int MT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tile_waves(MT)))) factor_trace_kernel(CalcArgs a)
{
    const int lane = threadIdx.x;
    const int nt = a.ntypes;
    const int bnode = (int)(blockIdx.x / nt);
    const int t = (int)(blockIdx.x - (unsigned)bnode * nt);
    if (bnode >= a.nbatch)
        return;
    const int node = a.node_list ? a.node_list[a.node0 + bnode] : a.node0 + bnode;
    const int m = a.m;
    const int pt = a.counts[(size_t)node * nt + t];
    const size_t o = (size_t)t * a.nnode + node;
    if (pt == 0) {
        if (lane == 0) {
            a.pnlobs[o] = 0;
            a.pdfs[o] = 0.0f;
            a.psrf[o] = 0.0f;
        }
        return;
    }
    if (lane == 0)
        a.pnlobs[o] = pt;
    // every local obs of the node is of this type: M_t is the node's own M,
    // whose diagnostics the node's kernel (earlier on this stream) has
    // written; the reference's re-solve works on the same matrix
    const long long p = a.offsets[(size_t)(node + 1) * nt] - a.offsets[(size_t)node * nt];
    if (pt == p) {
        if (lane == 0) {
            const size_t ot = (size_t)nt * a.nnode + node;
            const float fd = a.pdfs[ot];
            a.pdfs[o] = fd;
            a.psrf[o] = ((double)fd > kDfsMin) ? a.psrf[ot] : 0.0f;
        }
        return;
    }
    tile4 x[tri_count(MT)];
    const double trg = load_tiles<MT, true>(a, bnode, node, t, t + 1, lane, x);
    bool bad = false;
    float log2det;
    tile_eliminate<MT>(x, lane, bad, log2det);
    tile_invert_factor<MT>(x, lane);
    if (__ballot(bad) && lane == 0)
        atomicExch(a.err, ENKFG_ERR_LINALG);
    // tr(M^-1) = |V|^2
    double s = 0.0;
#pragma unroll
    for (int f = 0; f < tri_count(MT); ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            s = fma(x[f][r], x[f][r], s);
    s = wave_sum(s) - (double)(16 * MT - m);
    if (lane == 0) {
        const float fd = (float)((double)m - s);
        a.pdfs[o] = fd;
        a.psrf[o] = ((double)fd > kDfsMin) ? (float)(sqrt(trg / (double)fd) - 1.0) : 0.0f;
    }
}

// ADJ: z = M^-1 g and w = M^-1 S^T s per listed node, and M^-1 itself
template <int MT, bool ADJ>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tile_waves(MT)))) factor_tile_kernel(CalcArgs a)
{
    constexpr int MP = 16 * MT;
    __shared__ TileLds<MT> sh;
    const int lane = threadIdx.x;
    const int nt = a.ntypes;
    const int bnode = (int)blockIdx.x;
    if (bnode >= a.nbatch)
        return;
    const int node = a.node_list ? a.node_list[a.node0 + bnode] : a.node0 + bnode;
    const int m = a.m, md = a.md;
    const bool dotT = a.mode == ENKFG_MODE_ENKF || a.mode == ENKFG_MODE_HYBRID;
    const long long off = a.offsets[(size_t)node * nt];
    const int p = (int)(a.offsets[(size_t)(node + 1) * nt] - off);
    const size_t lk = (size_t)(a.node0 + bnode);   // adjoint: index in the node list
    if (ADJ && p == 0) {
        for (int e = lane; e < m; e += 64) {
            a.adj_z[lk * m + e] = 0.0;
            a.adj_w[lk * m + e] = 0.0;
        }
        if (a.adj_minv != nullptr)   // no local obs: T = I whatever M (nothing depends on it)
            for (int k = lane; k < MP * MP; k += 64)
                a.adj_minv[(size_t)bnode * MP * MP + k] = 0.0;
        return;
    }
    if (!ADJ) {
        if (!a.pertype)
            for (int t = lane; t < nt; t += 64) {
                a.pnlobs[(size_t)t * a.nnode + node] = a.counts[(size_t)node * nt + t];
                a.pdfs[(size_t)t * a.nnode + node] = 0.0f;
                a.psrf[(size_t)t * a.nnode + node] = 0.0f;
            }
        if (p == 0) {
            if (lane == 0) {
                a.pnlobs[(size_t)nt * a.nnode + node] = 0;
                a.pdfs[(size_t)nt * a.nnode + node] = 0.0f;
                a.psrf[(size_t)nt * a.nnode + node] = 0.0f;
            }
            // empty column: T = I, w = 0 (transforms.c:766-780)
            if (dotT)
                for (int k = lane; k < md * m; k += 64) {
                    const int e1 = k / m, e2 = k - e1 * m;
                    a.T[(size_t)node * md * m + k] = (e1 == e2) ? 1.0f : 0.0f;
                    if (a.T64 != nullptr)
                        a.T64[(size_t)node * md * m + k] = (e1 == e2) ? 1.0 : 0.0;
                }
            for (int e = lane; e < m; e += 64) {
                a.w[(size_t)node * m + e] = 0.0f;
                if (a.w64 != nullptr)
                    a.w64[(size_t)node * m + e] = 0.0;
            }
            return;
        }
    }
    tile4 x[tri_count(MT)];
    const double trg = load_tiles<MT, ADJ>(a, bnode, node, 0, a.nseg, lane, x);
    // S^T s over the segments
    for (int e = lane; e < MP; e += 64) {
        double v = 0.0;
        if (e < m)
            for (int s = 0; s < a.nseg; ++s)
                if (!a.pertype || a.counts[(size_t)node * nt + s] != 0)
                    v += a.sts[((size_t)bnode * a.nseg + s) * MP + e];
        sh.b[e] = v;
        if (ADJ)
            sh.g[e] = e < m ? a.adj_g[(size_t)node * m + e] : 0.0;
    }
    __syncthreads();
    bool bad = false;
    float log2det;
    tile_eliminate<MT>(x, lane, bad, log2det);
    tile_invert_factor<MT>(x, lane);
    if (__ballot(bad) && lane == 0)
        atomicExch(a.err, ENKFG_ERR_LINALG);

#pragma unroll
    for (int f = 0; f < tri_count(MT); ++f)
        tile_pin(x[f]);

    // M^-1, a tile and its transpose written as soon as it is known; yb[e] =
    // (M^-1 b) from this lane's rows of column block e (yg: of g)
    const int col = lane & 15, grp = lane >> 4;
    double yb[MT], yg[ADJ ? MT : 1];
    double trx = 0.0;
#pragma unroll
    for (int k = 0; k < MT; ++k)
        yb[k] = 0.0;
    if (ADJ)
#pragma unroll
        for (int k = 0; k < (ADJ ? MT : 1); ++k)
            yg[k] = 0.0;
    // rows of T (adjoint: of M^-1) to write, in FP32 and FP64
    const int tlim = dotT ? md : 0;
    const int tlim64 = ADJ ? (a.adj_minv != nullptr ? MP : 0) : (dotT && a.T64 != nullptr ? md : 0);
    auto put = [&](auto ic, auto jc, const tile4& v) {   // tile (I, J) of M^-1
        constexpr int I = ic, J = jc;
        // the lane's place, opaque in each tile: what is derived from it is
        // formed where it is used, and the tiles are taken one after another,
        // so that neither takes registers from the tiles
        // (and the row limits opaque, or the compiler makes a copy of the
        // kernel for each case)
        int col = lane & 15, grp = lane >> 4, t32 = tlim, t64 = tlim64;
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(col), "+v"(grp), "+s"(t32), "+s"(t64));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e1 = 16 * I + 4 * r + grp, e2 = 16 * J + col;
            if (ADJ) {
                if (e1 < t64)
                    a.adj_minv[((size_t)bnode * MP + e1) * MP + e2] = (e1 < m && e2 < m) ? v[r] : 0.0;
            } else {
                const double dlt = (e1 == e2) ? 1.0 : 0.0;
                double t = 0.5 * v[r] + 0.5 * dlt;
                t = (t - dlt) * a.alpha + dlt;
                const size_t o = ((size_t)node * md + e1) * m + e2;
                if (e1 < t32 && e2 < m)
                    a.T[o] = (float)t;
                if (e1 < t64 && e2 < m)
                    a.T64[o] = t;
            }
        }
        double y = 0.0, z = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            y = fma(v[r], sh.b[16 * I + 4 * r + grp], y);
            if (ADJ)
                z = fma(v[r], sh.g[16 * I + 4 * r + grp], z);
        }
        // (here, not where yb is used, which would keep v and b)
        y += yb[J];
        asm volatile("" : "+v"(y));
        yb[J] = y;
        if (ADJ) {
            z += yg[ADJ ? J : 0];
            asm volatile("" : "+v"(z));
            yg[ADJ ? J : 0] = z;
        }
    };
    tile_inverse<MT>(x, [&](auto ic, auto jc, tile4& v) {
        constexpr int i = ic, j = jc;
        put(ic, jc, v);
        if constexpr (i == j) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                trx += (4 * r + grp == col) ? v[r] : 0.0;
            asm volatile("" : "+v"(trx));
        } else {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sh.t[4 * r + grp][col] = v[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] = sh.t[col][4 * r + grp];
            put(jc, ic, v);
        }
    });
    trx = wave_sum(trx) - (double)(MP - m);
    if (!ADJ && lane == 0) {
        const float fd = (float)((double)m - trx);   // m - tr(M^-1)
        a.pnlobs[(size_t)nt * a.nnode + node] = p;
        a.pdfs[(size_t)nt * a.nnode + node] = fd;
        a.psrf[(size_t)nt * a.nnode + node] = (float)(sqrt(trg / (double)fd) - 1.0);
    }
    // w (z): the columns' sums over the four row groups
#pragma unroll
    for (int k = 0; k < MT; ++k) {
        double y = yb[k];
        y += __shfl_xor(y, 16);
        y += __shfl_xor(y, 32);
        const int e = 16 * k + col;
        if (ADJ) {
            double z = yg[ADJ ? k : 0];
            z += __shfl_xor(z, 16);
            z += __shfl_xor(z, 32);
            if (grp == 0 && e < m) {
                a.adj_w[lk * m + e] = y;
                a.adj_z[lk * m + e] = z;
            }
        } else if (grp == 0 && e < m) {
            a.w[(size_t)node * m + e] = (float)y;
            if (a.w64 != nullptr)
                a.w64[(size_t)node * m + e] = y;
        }
    }
}

template <int MT>
hipError_t launch_mt(hipStream_t s, const CalcArgs& a)
{
    const dim3 grid((unsigned)a.nbatch);
    if (a.adj_g != nullptr) {
        if constexpr (MT <= 6)
            hipLaunchKernelGGL((factor_tile_kernel<MT, true>), grid, dim3(64), 0, s, a);
        else
            return hipErrorInvalidValue;
    } else {
        hipLaunchKernelGGL((factor_tile_kernel<MT, false>), grid, dim3(64), 0, s, a);
    }
    return hipGetLastError();
}

template <int MT>
void launch_trace_mt(hipStream_t s, const CalcArgs& a)
{
    hipLaunchKernelGGL(factor_trace_kernel<MT>, dim3((unsigned)((long long)a.nbatch * a.ntypes)), dim3(64), 0, s, a);
}

}  // namespace

bool factor_wave_supported(const CalcArgs& a)
{
    const bool etkf = a.scheme == ENKFG_SCHEME_ETKF && a.mode != ENKFG_MODE_ENOI;
    return !etkf && a.m <= 160;
}

hipError_t launch_factor_wave(hipStream_t s, const CalcArgs& a)
{
    if (a.nbatch == 0)
        return hipSuccess;
    hipError_t e;
    switch ((a.m + 15) / 16) {
    case 1: e = launch_mt<1>(s, a); break;
    case 2: e = launch_mt<2>(s, a); break;
    case 3: e = launch_mt<3>(s, a); break;
    case 4: e = launch_mt<4>(s, a); break;
    case 5: e = launch_mt<5>(s, a); break;
    case 6: e = launch_mt<6>(s, a); break;
    case 7: e = launch_mt<7>(s, a); break;
    case 8: e = launch_mt<8>(s, a); break;
    case 9: e = launch_mt<9>(s, a); break;
    case 10: e = launch_mt<10>(s, a); break;
    default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess || !a.pertype || a.adj_g != nullptr)
        return e;
    return launch_factor_trace(s, a);
}

hipError_t launch_factor_trace(hipStream_t s, const CalcArgs& a)
{
    if (a.nbatch == 0 || a.ntypes <= 0)
        return hipSuccess;
    // per-obstype diagnostics, one work item per (node, obstype)
    switch ((a.m + 15) / 16) {
    case 1: launch_trace_mt<1>(s, a); break;
    case 2: launch_trace_mt<2>(s, a); break;
    case 3: launch_trace_mt<3>(s, a); break;
    case 4: launch_trace_mt<4>(s, a); break;
    case 5: launch_trace_mt<5>(s, a); break;
    case 6: launch_trace_mt<6>(s, a); break;
    case 7: launch_trace_mt<7>(s, a); break;
    case 8: launch_trace_mt<8>(s, a); break;
    case 9: launch_trace_mt<9>(s, a); break;
    case 10: launch_trace_mt<10>(s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace enkfg
