// factor_etkf.hip -- the ETKF factorisation: T = M^-1/2, w, dfs and srf of a
// node, one wavefront per node, on 16 x 16 FP64 matrix-core tiles
// (tile_matrix.h).
//
// M^-1/2 comes from the scaled, coupled Denman-Beavers iteration (Higham,
// "Functions of Matrices", SIAM 2008, eq. 6.15 and sec. 6.3),
//   Z_{k+1} = (mu_k Z_k + Y_k^-1 / mu_k) / 2,   Z_0 = I   (-> M^-1/2)
//   Y_{k+1} = (mu_k Y_k + Z_k^-1 / mu_k) / 2,   Y_0 = M   (-> M^1/2)
//   mu_k = |det Y_k det Z_k|^(-1/(2m))
// whose two inverses are the block elimination of the DEnKF factorisation.
// Y_k = M Z_k, so det Z_k = det Y_k / det M and mu_k is known from Y_k alone (in
// single precision: any scaling near it converges as fast).  The padding (rows
// m ..) is kept the identity in Y and Z, as it is in M: scaled with the rest, it
// would enter the determinants, whose root is of order 2m, and for m <= 7 mu
// runs away.  Each inverse is combined tile by tile as it is formed.  The first step
// needs one inverse (Z_0 = I; it gives w, dfs = tr(M^-1 G) and srf too), the last one
// Y_k^-1 only.  Once a step changes Z by less than 1e-8 of its norm, one more
// unscaled step is taken and is the last (the iteration converges
// quadratically); no convergence in 60 steps is reported.
//
// Y, Z and the next Z (upper tiles) live in a workspace per wavefront; the
// registers hold the matrix that is being inverted.  Wavefronts loop over the
// batch's nodes, so the workspace is that of the resident ones.  Bound: the
// FP64 matrix cores (162 tile products an inverse for m = 96, 41k cycles) and
// the workspace's traffic (130 KB an inverse).  For m = 96 about 14 inverses
// a node.  Measured against the kernel before it (pivots swept one per
// workgroup barrier, one five-wave workgroup per CU): 51x1500x1800 tile FP64
// calc 1,909 -> 550 ms; 4,050 nodes, m = 96: 21.0 -> 3.9 ms; 2,278 nodes, m =
// 24: 0.61 -> 0.23 ms.  m > 96 had iterates in memory and Gauss-Jordan
// inverses of up to 2 KB of spills a lane; it takes the same path now (136 B
// of spills a lane at MT = 6, 440 and 964 at 9 and 10: tile_waves).
#include <algorithm>

#include "enkfg_internal.h"
#include "gram_layout.h"
#include "tile_matrix.h"

namespace enkfg {

namespace {

template <int MT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tile_waves(MT)))) factor_etkf_kernel(CalcArgs a)
{
    constexpr int MP = 16 * MT;
    constexpr size_t GS = gram_size(MT);
    __shared__ TileLds<MT> sh;
    const int nt = a.ntypes;
    const int m = a.m, md = a.md;
    double* const ws = a.etkf_ws + (size_t)blockIdx.x * etkf_ws_size(m);
    for (int bnode = (int)blockIdx.x; bnode < a.nbatch; bnode += (int)gridDim.x) {
        int lane = threadIdx.x;
        asm volatile("" : "+v"(lane));   // (nothing formed from it is kept across the loop)
        const int node = a.node_list ? a.node_list[a.node0 + bnode] : a.node0 + bnode;
        const long long off = a.offsets[(size_t)node * nt];
        const int p = (int)(a.offsets[(size_t)(node + 1) * nt] - off);
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
            continue;
        }
        __syncthreads();   // (the previous node's reads of sh.b)
        for (int e = lane; e < MP; e += 64) {
            double v = 0.0;
            if (e < m)
                for (int s = 0; s < a.nseg; ++s)
                    if (!a.pertype || a.counts[(size_t)node * nt + s] != 0)
                        v += a.sts[((size_t)bnode * a.nseg + s) * MP + e];
            sh.b[e] = v;
        }
        __syncthreads();

        // Y_0 = M
        double trg, g2;
        {
            tile4 x[tri_count(MT)];
            trg = load_tiles<MT, false, true>(a, bnode, node, 0, a.nseg, lane, x, &g2);
#pragma unroll
            for (int f = 0; f < tri_count(MT); ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    ws[f * 256 + 64 * r + lane] = x[f][r];
        }
        // inverse number ph: of M (ph 0), then of Y (odd) and Z (even) in turn
        int zi = 0;   // Z is buffer zi
        bool bad = false, last = false, done = false;
        float ldM = 0.0f;
        double mu = 1.0;
        int ph = 0;
        for (; ph < 120; ++ph) {
            // the lane and the buffers, opaque in each pass: the masks and
            // addresses formed from them are not kept across the loop
            int lane = threadIdx.x;
            const int zu = __builtin_amdgcn_readfirstlane(zi);
            unsigned oz = (unsigned)(1 + zu) * (unsigned)GS, on = (unsigned)(2 - zu) * (unsigned)GS, oy = 0;
            asm volatile("" : "+v"(lane), "+s"(oy), "+s"(oz), "+s"(on));
            double* Y = ws + oy;
            double* Z = ws + oz;
            double* Zn = ws + on;
            const bool first = ph == 0;
            const bool ofY = first || (ph & 1) != 0;   // the inverse goes into Z
            tile4 x[tri_count(MT)];
            // diagonal tiles are read as other lanes of this wavefront stored them
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            read_tiles<MT, 0, tri_count(MT)>(ofY ? Y : Z, lane, x);
#pragma unroll
            for (int f = 0; f < tri_count(MT); ++f)
                tile_pin(x[f]);
            float log2det;
            tile_eliminate<MT>(x, lane, bad, log2det);
            tile_invert_factor<MT>(x, lane);
#pragma unroll
            for (int f = 0; f < tri_count(MT); ++f)
                tile_pin(x[f]);
            if (first)
                ldM = log2det;
            if (ofY)
                mu = last ? 1.0 : (double)__builtin_amdgcn_exp2f((ldM - 2.0f * log2det) / (float)(2 * m));
            // the tiles of the inverse (v), combined: Zn = (mu Z + v / mu) / 2, or
            // Y likewise in place
            const double hm = 0.5 * mu, hi = 0.5 * recip_pivot(mu);
            const double* other = ofY ? Z : Y;
            double* dst = ofY ? Zn : Y;
            const int fz = __builtin_amdgcn_readfirstlane(first ? 1 : 0);
            const int ft = __builtin_amdgcn_readfirstlane((last && ofY) ? 1 : 0);
            double yb[MT];
            double trx = 0.0, dn = 0.0, nn = 0.0;
#pragma unroll
            for (int k = 0; k < MT; ++k)
                yb[k] = 0.0;
            // sums of the first inverse with S^T s
            auto mulb = [&](auto ic, auto jc, const tile4& v) {
                constexpr int I = ic, J = jc;
                double y = yb[J];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    y = fma(v[r], sh.b[16 * I + 4 * r + (lane >> 4)], y);
                asm volatile("" : "+v"(y));
                yb[J] = y;
            };
            // rows of T = Z, relaxation T <- (T - I) alpha + I, FP32
            auto putT = [&](auto ic, auto jc, const tile4& v) {
                constexpr int I = ic, J = jc;
                int col = lane & 15, grp = lane >> 4, t64 = a.T64 != nullptr ? md : 0;
                asm volatile("" : "+v"(col), "+v"(grp), "+s"(t64));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int e1 = 16 * I + 4 * r + grp, e2 = 16 * J + col;
                    const double dlt = (e1 == e2) ? 1.0 : 0.0;
                    const double t = (v[r] - dlt) * a.alpha + dlt;
                    const size_t o = ((size_t)node * md + e1) * m + e2;
                    if (e1 < md && e2 < m)
                        a.T[o] = (float)t;
                    if (e1 < t64 && e2 < m)
                        a.T64[o] = t;
                }
            };
            auto transposed = [&](const tile4& v) {
                tile4 t;
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sh.t[4 * r + (lane >> 4)][lane & 15] = v[r];
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    t[r] = sh.t[lane & 15][4 * r + (lane >> 4)];
                return t;
            };
            auto put = [&](auto ic, auto jc, const tile4& v) {   // tile (I, J), I <= J
                constexpr int I = ic, J = jc;
                constexpr size_t at = (size_t)tri_at<MT>(I, J) * 256;
                int l0 = lane, z = fz, tt = ft;
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" : "+v"(l0), "+s"(z), "+s"(tt));
                tile4 o, eye, nv;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    eye[r] = (I == J && 4 * r + (l0 >> 4) == (l0 & 15)) ? 1.0 : 0.0;
                // the last diagonal tile's columns m .. (elsewhere theirs stay 0)
                const bool pad = I == J && I == MT - 1 && 16 * I + (l0 & 15) >= m;
                if (z) {
                    o = eye;
                    // Y_1 = (mu M + I / mu) / 2
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        Y[at + 64 * r + l0] = pad ? eye[r] : hm * Y[at + 64 * r + l0] + hi * eye[r];
                    mulb(ic, jc, v);
                    if (I == J) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            trx += eye[r] * v[r];
                    } else {
                        mulb(jc, ic, transposed(v));
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        o[r] = other[at + 64 * r + l0];
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    nv[r] = pad ? eye[r] : hm * o[r] + hi * v[r];
                    const double d = nv[r] - o[r];
                    // off-diagonal tiles stand for themselves and their transposes
                    dn += (I == J ? 1.0 : 2.0) * d * d;
                    nn += pad ? 0.0 : (I == J ? 1.0 : 2.0) * nv[r] * nv[r];
                }
                asm volatile("" : "+v"(dn), "+v"(nn), "+v"(trx));
                if (tt) {
                    putT(ic, jc, nv);
                    if (I != J)
                        putT(jc, ic, transposed(nv));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        dst[at + 64 * r + l0] = nv[r];
                }
            };
            tile_inverse<MT>(x, [&](auto ic, auto jc, const tile4& v) { put(ic, jc, v); });
            if (first) {
                trx = wave_sum(trx) - (double)(MP - m);
                if (lane == 0) {
                    // m - tr(M^-1) to m eps; where that shows, by the first two
                    // terms of tr(G) - tr(G^2) + tr(G^3) - ..., to 1e-10
                    const double dfs = (double)m - trx;
                    const float fd = (float)(dfs > 1e-5 ? dfs : trg - g2);
                    a.pnlobs[(size_t)nt * a.nnode + node] = p;
                    a.pdfs[(size_t)nt * a.nnode + node] = fd;
                    a.psrf[(size_t)nt * a.nnode + node] = (float)(sqrt(trg / (double)fd) - 1.0);
                }
#pragma unroll
                for (int k = 0; k < MT; ++k) {
                    double y = yb[k];
                    y += __shfl_xor(y, 16);
                    y += __shfl_xor(y, 32);
                    const int e = 16 * k + (lane & 15);
                    if (lane < 16 && e < m) {
                        a.w[(size_t)node * m + e] = (float)y;
                        if (a.w64 != nullptr)
                            a.w64[(size_t)node * m + e] = y;
                    }
                }
            }
            if (first) {   // Z_1 and Y_1 are there
                zi ^= 1;
                continue;
            }
            if (ofY) {
                done = last;
                if (last)
                    break;
                dn = wave_sum(dn);
                nn = wave_sum(nn);
                if (__ballot(dn <= 1e-16 * nn) != 0)   // (the same in every lane)
                    last = true;
            } else {       // Y_{k+1} is there: on to Z_{k+1}
                zi ^= 1;
            }
        }
        if ((!done || __ballot(bad)) && lane == 0)
            atomicExch(a.err, ENKFG_ERR_LINALG);   // no convergence, or a non-positive pivot
    }
}

template <int MT>
void launch_etkf_mt(hipStream_t s, const CalcArgs& a, int grid)
{
    hipLaunchKernelGGL(factor_etkf_kernel<MT>, dim3((unsigned)grid), dim3(64), 0, s, a);
}

}  // namespace

int etkf_groups(int m, int nbatch)
{
    // the wavefronts that 256 CUs of four SIMDs hold at once
    return std::min(nbatch, 1024 * tile_waves((m + 15) / 16));
}

hipError_t launch_factor_etkf(hipStream_t s, const CalcArgs& a)
{
    if (a.nbatch == 0)
        return hipSuccess;
    const int g = etkf_groups(a.m, a.nbatch);
    switch ((a.m + 15) / 16) {
    case 1: launch_etkf_mt<1>(s, a, g); break;
    case 2: launch_etkf_mt<2>(s, a, g); break;
    case 3: launch_etkf_mt<3>(s, a, g); break;
    case 4: launch_etkf_mt<4>(s, a, g); break;
    case 5: launch_etkf_mt<5>(s, a, g); break;
    case 6: launch_etkf_mt<6>(s, a, g); break;
    case 7: launch_etkf_mt<7>(s, a, g); break;
    case 8: launch_etkf_mt<8>(s, a, g); break;
    case 9: launch_etkf_mt<9>(s, a, g); break;
    case 10: launch_etkf_mt<10>(s, a, g); break;
    default: return hipErrorInvalidValue;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !a.pertype)
        return e;
    return launch_factor_trace(s, a);   // per-type diagnostics, after the node's own
}

}  // namespace enkfg
