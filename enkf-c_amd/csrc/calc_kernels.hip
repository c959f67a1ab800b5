// calc_kernels.hip -- per-column ensemble transforms for the FP64 path.
//
// For each stride-grid node the reference (calc/transforms.c:794-879 and
// calc/calcs.c) gathers the local standardised anomalies S (p x m, tapered,
// FP64), forms M = I + S^T S, factorises it and builds G = M^-1 S^T (m x p),
// T and w.  Here the p x m matrices are never formed:
//
//   gram   (MFMA FP64)  G0 = S^T S and S^T s, streamed from the gathered
//                       FP32 rows of S, tapered in FP64 on their way to LDS;
//   factor              M = I + G0 inverted, then (factor_tile.hip: DEnKF and
//                       EnOI; factor_etkf.hip: ETKF)
//                         T = (I + M^-1) / 2, or M^-1/2 (= I - (M+M^1/2)^-1 S^T S)
//                         w = M^-1 S^T s,  dfs = tr(M^-1 G0) (= tr(G S)),
//                         srf = sqrt(tr(G0) / dfs) - 1
//                       followed by relaxation to prior and the FP32 cast.
//
// The identities used are those of the User Guide (doc/enkf-userguide.tex:
// 440-451, 490-522); the per-type diagnostics, which re-solve the analysis
// with only the obs of one type as the USE_MPIQUEUE build does
// (transforms.c:853-879), are factor_tile.hip's factor_trace_kernel for
// every scheme.
#include <algorithm>

#include "enkfg_internal.h"
#include "gram_layout.h"
#include "gram_stage.h"

namespace enkfg {

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ utilities
__global__ void standardise_kernel(int nmem, int nobs, const short* __restrict__ type,
                                   const float* __restrict__ estd, const double* __restrict__ sqrt_rfactor,
                                   double mult, float* __restrict__ S, double* __restrict__ sv)
{
    // calc/ensobs.c:849-898: S /= estd * sqrt(rfactor) * sqrt(m - 1)
    const long long n = (long long)nobs * nmem;
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x) {
        const long long o = k / nmem;
        const double div = (double)estd[o] * sqrt_rfactor[type[o]] * mult;
        S[k] = (float)((double)S[k] / div);
        if (sv != nullptr && k % nmem == 0)
            sv[o] = sv[o] / div;
    }
}

__global__ void transpose_kernel(const float* __restrict__ in, float* __restrict__ out, long long rows, long long cols)
{
    __shared__ float tile[32][33];
    const long long c0 = (long long)blockIdx.x * 32, r0 = (long long)blockIdx.y * 32;
    for (int k = threadIdx.y; k < 32; k += 8) {
        long long r = r0 + k, c = c0 + threadIdx.x;
        if (r < rows && c < cols)
            tile[k][threadIdx.x] = in[r * cols + c];
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        long long c = c0 + k, r = r0 + threadIdx.x;
        if (r < rows && c < cols)
            out[c * rows + r] = tile[threadIdx.x][k];
    }
}

// Gather: dst row r (stride `stride`) = src row perm[r] (stride `width`)
// for r < nrow, zero padded to the stride, followed by one zero row.
// Scatter: dst row perm[r] (stride `width`) = the first `width` elements of
// src row r (stride `stride`).
template <class T, bool SCATTER>
__global__ void permute_rows_kernel(const T* __restrict__ src, const int* __restrict__ perm, T* __restrict__ dst,
                                    long long nrow, int width, int stride)
{
    const long long n = (SCATTER ? nrow : nrow + 1) * stride;
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x) {
        const long long r = k / stride;
        const int c = (int)(k - r * stride);
        if (SCATTER) {
            if (c < width)
                dst[(long long)perm[r] * width + c] = src[k];
        } else {
            dst[k] = (r < nrow && c < width) ? src[(long long)perm[r] * width + c] : T(0);
        }
    }
}

// ------------------------------------------------------------------ Gram, independent wavefronts
//
// Each wavefront computes one group of upper-triangle 16 x 16 tiles (tiles
// f = g, g + NG, ... of tri_count(MT); NG = 1 or 2 for m = 96, 4 or 5 groups
// of the 45 tiles for m = 144: item_groups_lo, chosen per obs-count bucket
// by the host's autotuner) of one (node, obstype segment), with no workgroup
// barrier: the wave stages its own chunks of IKC local obs through a private
// LDS area.  Per chunk: the copies of chunks c+1 and c+2 and the list
// entries of chunk c+3 are in flight while chunk c feeds the MFMAs.  The
// taper is applied in FP64 as an operand is formed, (double) S * lc, as the
// reference forms Sloc.
//
// Bound: the FP64 matrix cores (71.7 TFLOP/s in a large library product on
// this card).  51x1500x1800 tile, 1.771e13 flop: 47 TFLOP/s with two groups
// and a chunk's conversions ahead of its MFMAs, 56 with one group and the
// conversions between them, with the factor kernels of the previous batch
// running beside (calc 412 -> 379 ms).
// obs per chunk (kChunk, gram_stage.h): four k-steps.  With
// register-staged chunks, 16 rather than 8 gave a calc pass on the tile of
// 888 instead of 904 ms: at 8 the Gram took so many waves per CU that the
// factor kernels of the previous batch, on the other stream, overlapped it
// worse (32: 984 ms, 222 VGPRs).
constexpr int IKC = kChunk;
// chunk buffers (four measured 712.7 against 679.9 ms: six waves per CU)
constexpr int IKB = 3;
static_assert(kListPad >= (IKB + 2) * IKC, "list padding too small for the item Gram pipeline");
template <int MT>
using ItemLds = ChunkLds<MT, IKB>;

// number of tiles of group G of NG
template <int MT, int NG, int G>
constexpr int item_ntile()
{
    return (tri_count(MT) - G + NG - 1) / NG;
}

// the tiles f = G + NG t of group G: acc[t] += frag[I] frag[J]^T
template <int MT, int NG, int G, int T>
__device__ __attribute__((always_inline)) inline void item_tiles(const double (&frag)[MT], dbl4* acc)
{
    if constexpr (G + NG * T < tri_count(MT)) {
        constexpr int f = G + NG * T;
        constexpr int I = tri_I(MT, f), J = tri_J(MT, f);
        acc[T] = __builtin_amdgcn_mfma_f64_16x16x4f64(frag[I], frag[J], acc[T], 0, 0, 0);
        item_tiles<MT, NG, G, T + 1>(frag, acc);
    }
}

template <int MT, int NG, int G>
__device__ __attribute__((always_inline)) inline void item_wave(const CalcArgs& a, int b, long long off, int cnt, ItemLds<MT>& sh)
{
    constexpr int MP = 16 * MT;
    constexpr int NTG = item_ntile<MT, NG, G>();
    const int lane = threadIdx.x & 63;
    const int kq = lane >> 4;
    const int col = lane & 15;

    dbl4 acc[NTG > 0 ? NTG : 1];
#pragma unroll
    for (int f = 0; f < NTG; ++f)
        acc[f] = dbl4{0.0, 0.0, 0.0, 0.0};
    double sts[MT];
#pragma unroll
    for (int X = 0; X < MT; ++X)
        sts[X] = 0.0;

    // One k-step (four obs) ahead: while the matrix cores work on the
    // operands of step s, the lane reads, converts and tapers those of step
    // s + 1, its instructions interleaved with the MFMAs (in a wave's program
    // order all conversions of a chunk came first, then 44 MFMAs: 73% of the
    // matrix cores' time).  The last step of a chunk reads the next chunk's
    // first rows, whose copies chunk_advance waits for; by then every row of
    // the chunk itself has been read.
    const int nchunk = (cnt + IKC - 1) / IKC;
    chunk_prologue<MT, IKB>(a, sh, off, cnt);
    int buf = 0;    // c % IKB
    int slot = 0;   // c % (IKB + 1)
    double frag[MT], sl;
    auto operands = [&](int c, int b2, int sl2, int s, double (&f)[MT], double& t) {
        const int r = 4 * s + kq;
        const double lr = reinterpret_cast<const double*>(&sh.meta[sl2][16])[r];
        const double sv = reinterpret_cast<const double*>(&sh.sv[b2][0])[r];
        float raw[MT];
#pragma unroll
        for (int X = 0; X < MT; ++X)
            raw[X] = sh.rows[b2][X][r][col];
        const double l = c * IKC + r < cnt ? lr : 0.0;
#pragma unroll
        for (int X = 0; X < MT; ++X)
            f[X] = (double)raw[X] * l;
        t = sv * l;
    };
    chunk_advance<MT, IKB>(a, sh, off, cnt, 0, buf, slot);
    operands(0, 0, 0, 0, frag, sl);
    for (int c = 0; c < nchunk; ++c) {
        const int nbuf = buf == IKB - 1 ? 0 : buf + 1;
        const int nslot = slot == IKB ? 0 : slot + 1;
#pragma unroll
        for (int s = 0; s < IKC / 4; ++s) {
            double fn[MT], sn;
            if (s == IKC / 4 - 1) {
                chunk_fence();
                chunk_advance<MT, IKB>(a, sh, off, cnt, c + 1, nbuf, nslot);
                operands(c + 1, nbuf, nslot, 0, fn, sn);
            } else {
                operands(c, buf, slot, s + 1, fn, sn);
            }
            item_tiles<MT, NG, G, 0>(frag, acc);
            if (G == 0) {
#pragma unroll
                for (int X = 0; X < MT; ++X)
                    sts[X] += frag[X] * sl;
            }
            // the LDS reads, then a conversion or product after each MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, MT + 2, 0);
#pragma unroll
            for (int t = 0; t < NTG; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (4 * MT + 8 + NTG - 1) / NTG, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int X = 0; X < MT; ++X)
                frag[X] = fn[X];
            sl = sn;
        }
        buf = nbuf;
        slot = nslot;
    }
    // the copies of the chunks past the end land before the wave ends
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the accumulators as they stand (register i of lane l holds
    // D[4 i + l / 16][l % 16])
    double* gout = a.gram + (size_t)b * gram_size(MT) + lane;
#pragma unroll
    for (int t = 0; t < NTG; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            gout[(G + NG * t) * 256 + 64 * i] = acc[t][i];
    if (G == 0) {
        double* stsout = a.sts + (size_t)b * MP;
#pragma unroll
        for (int X = 0; X < MT; ++X) {
            double v = sts[X];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (kq == 0)
                stsout[16 * X + col] = v;
        }
    }
}

// wave of group g (the groups with no tile do nothing)
template <int MT, int NG, int G>
__device__ __attribute__((always_inline)) inline void item_dispatch(int g, const CalcArgs& a, int b, long long off,
                                                                    int cnt, ItemLds<MT>& sh)
{
    if constexpr (G < NG) {
        if (g == G) {
            if constexpr (item_ntile<MT, NG, G>() > 0)
                item_wave<MT, NG, G>(a, b, off, cnt, sh);
        } else {
            item_dispatch<MT, NG, G + 1>(g, a, b, off, cnt, sh);
        }
    }
}

// item `it` = (segment b, group g) of the batch
template <int MT, int NG>
__device__ __attribute__((always_inline)) inline void item_run(const CalcArgs& a, int it, ItemLds<MT>& sh)
{
    const ItemRef r = item_ref(a, it, NG);
    const int g = r.g, seg = r.seg;
    const int b = r.bn * a.nseg + seg;   // the (node, segment) slot of the Gram scratch
    const int node = a.node_list ? a.node_list[a.node0 + r.bn] : a.node0 + r.bn;
    long long off;
    int cnt;
    if (a.pertype) {
        off = a.offsets[(size_t)node * a.ntypes + seg];
        cnt = a.counts[(size_t)node * a.ntypes + seg];
    } else {
        off = a.offsets[(size_t)node * a.ntypes];
        cnt = (int)(a.offsets[(size_t)(node + 1) * a.ntypes] - off);
    }
    if (cnt > 0)
        item_dispatch<MT, NG, 0>(g, a, b, off, cnt, sh);
}

template <int MT, int NG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) gram_item_kernel(CalcArgs a)
{
    // one item per wave.  Blocks are handed out as earlier ones finish (the
    // hardware dispatcher is the work queue); each XCD takes runs of
    // kItemRun consecutive (segment, group) items, the NG groups of a
    // segment adjacent, so neighbouring nodes and the groups of one segment
    // share that XCD's L2
    __shared__ ItemLds<MT> sh;
    const int nitem = a.nbatch * a.nseg * NG;
    const int it = item_of_block();
    if (it < nitem)
        item_run<MT, NG>(a, it, sh);
}

}  // namespace

hipError_t launch_standardise(hipStream_t s, int nmem, int nobs, const short* type, const float* estd,
                              const double* sqrt_rfactor, float* S_obsmajor, double* sv)
{
    const long long n = (long long)nmem * nobs;
    if (n == 0)
        return hipSuccess;
    const double mult = sqrt((double)nmem - 1);
    long long nb = (n + 255) / 256;
    if (nb > 65536)
        nb = 65536;
    hipLaunchKernelGGL(standardise_kernel, dim3((unsigned)nb), dim3(256), 0, s, nmem, nobs, type, estd, sqrt_rfactor,
                       mult, S_obsmajor, sv);
    return hipGetLastError();
}

hipError_t launch_transpose_f32(hipStream_t s, const float* in, float* out, long long rows, long long cols)
{
    if (rows == 0 || cols == 0)
        return hipSuccess;
    dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32));
    if (grid.y > 65535)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(transpose_kernel, grid, dim3(32, 8), 0, s, in, out, rows, cols);
    return hipGetLastError();
}

template <class T, bool SCATTER>
hipError_t launch_permute(hipStream_t s, const T* src, const int* perm, T* dst, long long nrow, int width, int stride)
{
    const long long n = (SCATTER ? nrow : nrow + 1) * stride;
    if (n == 0)
        return hipSuccess;
    const long long nb = std::min<long long>((n + 255) / 256, 65536);
    hipLaunchKernelGGL((permute_rows_kernel<T, SCATTER>), dim3((unsigned)nb), dim3(256), 0, s, src, perm, dst, nrow,
                       width, stride);
    return hipGetLastError();
}

hipError_t launch_gather_rows(hipStream_t s, const float* src, const int* perm, float* dst, long long nrow, int width,
                              int stride)
{
    return launch_permute<float, false>(s, src, perm, dst, nrow, width, stride);
}
hipError_t launch_gather_rows(hipStream_t s, const double* src, const int* perm, double* dst, long long nrow,
                              int width, int stride)
{
    return launch_permute<double, false>(s, src, perm, dst, nrow, width, stride);
}
hipError_t launch_scatter_rows(hipStream_t s, const float* src, const int* perm, float* dst, long long nrow, int width,
                               int stride)
{
    return launch_permute<float, true>(s, src, perm, dst, nrow, width, stride);
}
hipError_t launch_scatter_rows(hipStream_t s, const double* src, const int* perm, double* dst, long long nrow,
                               int width, int stride)
{
    return launch_permute<double, true>(s, src, perm, dst, nrow, width, stride);
}

template <int M>
void launch_gram_item(hipStream_t s, dim3 grid, const CalcArgs& a, int ng)
{
    constexpr int lo = item_groups_lo(M);
    if (ng == item_groups_many(M))
        hipLaunchKernelGGL((gram_item_kernel<M, item_groups_many(M)>), grid, dim3(64), 0, s, a);
    else if (ng == lo)
        hipLaunchKernelGGL((gram_item_kernel<M, lo>), grid, dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL((gram_item_kernel<M, lo + 1>), grid, dim3(64), 0, s, a);
}

hipError_t launch_gram(hipStream_t s, const CalcArgs& a)
{
    const int MT = (a.m + 15) / 16;
    if (a.nbatch == 0)
        return hipSuccess;
    if (MT < 1 || MT > 10)
        return hipErrorInvalidValue;
    // tile groups per segment: one of the two candidates of this MT (the
    // larger by default)
    const int lo = item_groups_lo(MT);
    const long long nlist = (long long)a.nbatch * a.nseg;
    const int ng = few_lists(MT, nlist) ? item_groups_many(MT) : (a.tile_groups == lo ? lo : lo + 1);
    const long long nitem = (long long)a.nbatch * a.nseg * ng;
    const dim3 igrid(item_grid(nitem));
    switch (MT) {
    case 1: launch_gram_item<1>(s, igrid, a, ng); break;
    case 2: launch_gram_item<2>(s, igrid, a, ng); break;
    case 3: launch_gram_item<3>(s, igrid, a, ng); break;
    case 4: launch_gram_item<4>(s, igrid, a, ng); break;
    case 5: launch_gram_item<5>(s, igrid, a, ng); break;
    case 6: launch_gram_item<6>(s, igrid, a, ng); break;
    case 7: launch_gram_item<7>(s, igrid, a, ng); break;
    case 8: launch_gram_item<8>(s, igrid, a, ng); break;
    case 9: launch_gram_item<9>(s, igrid, a, ng); break;
    default: launch_gram_item<10>(s, igrid, a, ng); break;
    }
    return hipGetLastError();
}

hipError_t launch_factor(hipStream_t s, const CalcArgs& a)
{
    // DEnKF and EnOI (factor_tile.hip), or ETKF (factor_etkf.hip)
    return factor_wave_supported(a) ? launch_factor_wave(s, a) : launch_factor_etkf(s, a);
}

}  // namespace enkfg
