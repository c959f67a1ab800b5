// gram_mixed.hip -- G0 = S^T S and S^T s of the local analyses in mixed
// precision: BF16 MFMA with FP32 accumulation on a hi/lo split of the tapered
// anomalies.
//
// Each tapered value x = S * (float) lc is split as x = hi + lo + r with
// hi = bf16(x), lo = bf16(x - hi) and |r| <= 2^-18 |x|; the product x_a x_b
// is taken as hi_a hi_b + hi_a lo_b + lo_a hi_b, which leaves out lo_a lo_b
// (<= 2^-18 relative), so every term of S^T S carries a relative error of
// about 2^-17 before the FP32 accumulation.  S^T s is summed from x, in FP32
// over four obs and in FP64 beyond.  The result is written in the FP64 Gram
// layout and the factorisation that follows stays in FP64 (factor_tile.hip).
//
// Work items, chunk pipeline and XCD placement are those of the FP64 item
// Gram kernel (calc_kernels.hip, gram_stage.h, gram_layout.h).
#include <algorithm>
#include <type_traits>

#include "enkfg_internal.h"
#include "gram_layout.h"
#include "gram_stage.h"

namespace enkfg {

namespace {

typedef float flt4 __attribute__((__vector_size__(4 * sizeof(float))));

// ------------------------------------------------------------------ one wavefront per work item
//
// For m <= 160: independent wavefronts, no workgroup barrier.  A wavefront
// computes one of NG groups of the tri_count(MT) tiles (f = g, g + NG, ...;
// NG = 1 or 2 for m = 96: all 21 tiles, or 11 and 10, FP32 accumulators;
// NG is chosen per obs-count bucket by the host's autotuner) of one (node,
// obstype segment).  The segment's list entries and S rows are copied into
// the wave's private LDS area in chunks of kChunk = 16 local obs, MKB chunks
// deep, with no VGPRs held for data in flight (gram_stage.h, the same
// pipeline as the FP64 item kernel).  Two chunks make one K = 32 step of
// v_mfma_f32_16x16x32_bf16 (twice the rate of the K = 16 form on this card):
// lane (col, kg) forms its operand of block X -- obs 4 kg .. 4 kg + 3 of
// either chunk, member 16 X + col -- from FP32 values of the block-major rows,
// x = S * (float) lc, split into BF16 hi = bf16(x) and lo = bf16(x - hi) (the
// split carries about 2^-17 relative error); each element is converted once
// per wave.  S^T s is summed from x in FP32 over four obs and in FP64 beyond.
// Bound: VALU issue of the split (about 180 instructions a chunk beside 32
// MFMAs of 16 cycles for m = 96).  51x1500x1800 tile: mixed calc 201 ms with
// two wavefronts a list and K = 16, 156 with one, 145 with K = 32 and the
// operands of the next step formed between the MFMAs.
constexpr int MKB = 3;
static_assert(kListPad >= (MKB + 4) * kChunk, "list padding too small for the mixed item Gram pipeline");
template <int MT>
using MixItemLds = ChunkLds<MT, MKB>;
typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef float flt2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

template <int MT, int NG, int G>
constexpr int mix_item_ntile()
{
    return (tri_count(MT) - G + NG - 1) / NG;
}

// the schedule of half a step: the LDS reads, then the conversions between
// the MFMAs
template <int MT, int NM>
__device__ __attribute__((always_inline)) inline void mix_interleave()
{
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * MT + 8, 0);
    if constexpr (NM > 0) {
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (24 * MT + 30 + NM - 1) / NM, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
}

// the tiles f = G + NG t, T0 <= t < T1, of group G
template <int MT, int NG, int G, int T0, int T1>
__device__ __attribute__((always_inline)) inline void mix_item_tiles(const bf16x8 (&h)[MT], const bf16x8 (&l)[MT],
                                                                     flt4* acc)
{
    if constexpr (T0 < T1) {
        constexpr int f = G + NG * T0;
        constexpr int I = tri_I(MT, f), J = tri_J(MT, f);
        acc[T0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h[I], h[J], acc[T0], 0, 0, 0);
        acc[T0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h[I], l[J], acc[T0], 0, 0, 0);
        acc[T0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[I], h[J], acc[T0], 0, 0, 0);
        mix_item_tiles<MT, NG, G, T0 + 1, T1>(h, l, acc);
    }
}

template <int MT, int NG, int G>
__device__ __attribute__((always_inline)) inline void mix_item_wave(const CalcArgs& a, int b, long long off, int cnt,
                                                                    MixItemLds<MT>& sh)
{
    constexpr int MP = 16 * MT;
    constexpr int NTG = mix_item_ntile<MT, NG, G>();
    const int lane = threadIdx.x & 63;
    const int kg = lane >> 4;      // which 4 obs of a chunk
    const int col = lane & 15;

    flt4 acc[NTG > 0 ? NTG : 1];
#pragma unroll
    for (int f = 0; f < NTG; ++f)
        acc[f] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
    double sts[MT];
#pragma unroll
    for (int X = 0; X < MT; ++X)
        sts[X] = 0.0;

    const int nchunk = (cnt + kChunk - 1) / kChunk;
    chunk_prologue<MT, MKB>(a, sh, off, cnt);
    int buf = 0;    // c % MKB
    int slot = 0;   // c % (MKB + 1)
    const int k0 = 4 * kg;
    // The operands of a K = 32 step: lane l supplies 8 obs of member row
    // l % 16 of a tile, here 4 (l / 16) .. of chunk c (HALF 0) and of chunk
    // c + 1 (HALF 1); which obs is which k does not matter as both operands
    // agree.  Past the list's end rows and tapers are 0.
    auto form = [&](auto half, int c, bf16x8 (&h)[MT], bf16x8 (&l)[MT]) {
        constexpr int o = 4 * decltype(half)::value;
        const double* svc = reinterpret_cast<const double*>(&sh.sv[buf][0]);
        const double* lcc = reinterpret_cast<const double*>(&sh.meta[slot][16]);
        // tapers of the lane's 4 obs and s * lc
        float lcf[4], slv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double lr = lcc[k0 + q];
            const double lq = c * kChunk + k0 + q < cnt ? lr : 0.0;
            lcf[q] = (float)lq;
            slv[q] = (float)(svc[k0 + q] * lq);
        }
        // (pairs converted together: v_cvt_pk_bf16_f32)
#pragma unroll
        for (int X = 0; X < MT; ++X) {
            float t = 0.0f;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                flt2v x;
                x[0] = sh.rows[buf][X][k0 + 2 * p][col] * lcf[2 * p];
                x[1] = sh.rows[buf][X][k0 + 2 * p + 1][col] * lcf[2 * p + 1];
                const bf16x2v hp = __builtin_convertvector(x, bf16x2v);
                const flt2v r = x - __builtin_convertvector(hp, flt2v);
                const bf16x2v lp = __builtin_convertvector(r, bf16x2v);
                h[X][o + 2 * p] = hp[0];
                h[X][o + 2 * p + 1] = hp[1];
                l[X][o + 2 * p] = lp[0];
                l[X][o + 2 * p + 1] = lp[1];
                if (G == 0) {
                    t = fmaf(x[0], slv[2 * p], t);
                    t = fmaf(x[1], slv[2 * p + 1], t);
                }
            }
            if (G == 0)
                sts[X] += (double)t;
        }
    };
    auto next = [&](int c) {   // chunk c: its copies have landed, later ones are issued
        buf = buf == MKB - 1 ? 0 : buf + 1;
        slot = slot == MKB ? 0 : slot + 1;
        chunk_fence();
        chunk_advance<MT, MKB>(a, sh, off, cnt, c, buf, slot);
    };
    // operands one step (two chunks) ahead: while the matrix cores work on
    // this step's tiles, the lane forms the next step's operands, half of
    // them beside half of the tiles
    bf16x8 h[MT], l[MT];
    chunk_advance<MT, MKB>(a, sh, off, cnt, 0, 0, 0);
    form(std::integral_constant<int, 0>{}, 0, h, l);
    next(1);
    form(std::integral_constant<int, 1>{}, 1, h, l);
    constexpr int TH = (NTG + 1) / 2;
    for (int c = 0; c < nchunk; c += 2) {
        bf16x8 hn[MT], ln[MT];
        next(c + 2);
        form(std::integral_constant<int, 0>{}, c + 2, hn, ln);
        mix_item_tiles<MT, NG, G, 0, TH>(h, l, acc);
        mix_interleave<MT, 3 * TH>();
        next(c + 3);
        form(std::integral_constant<int, 1>{}, c + 3, hn, ln);
        mix_item_tiles<MT, NG, G, TH, NTG>(h, l, acc);
        mix_interleave<MT, 3 * (NTG - TH)>();
#pragma unroll
        for (int X = 0; X < MT; ++X) {
            h[X] = hn[X];
            l[X] = ln[X];
        }
    }
    // the copies of the chunks past the end land before the wave ends
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // v_mfma_f32_16x16x32_bf16 result: register i of lane l holds
    // D[4 (l / 16) + i][l % 16]
    double* gout = a.gram + (size_t)b * gram_size(MT) + 64 * kg + col;
#pragma unroll
    for (int t = 0; t < NTG; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            gout[(G + NG * t) * 256 + 16 * i] = (double)acc[t][i];
    if (G == 0) {
        // the four lanes of a member (kg = 0..3) hold partial sums over
        // their 4 obs of each chunk
        double* stsout = a.sts + (size_t)b * MP;
#pragma unroll
        for (int X = 0; X < MT; ++X) {
            double v = sts[X];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (kg == 0)
                stsout[16 * X + col] = v;
        }
    }
}

template <int MT, int NG, int G>
__device__ __attribute__((always_inline)) inline void mix_item_dispatch(int g, const CalcArgs& a, int b, long long off,
                                                                        int cnt, MixItemLds<MT>& sh)
{
    if constexpr (G < NG) {
        if (g == G) {
            if constexpr (mix_item_ntile<MT, NG, G>() > 0)
                mix_item_wave<MT, NG, G>(a, b, off, cnt, sh);
        } else {
            mix_item_dispatch<MT, NG, G + 1>(g, a, b, off, cnt, sh);
        }
    }
}

// item `it` = (segment b, group g) of the batch
template <int MT, int NG>
__device__ __attribute__((always_inline)) inline void mix_item_run(const CalcArgs& a, int it, MixItemLds<MT>& sh)
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
        mix_item_dispatch<MT, NG, 0>(g, a, b, off, cnt, sh);
}

template <int MT, int NG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) gram_mixed_item_kernel(CalcArgs a)
{
    // one item per wave.  Blocks are handed out as earlier ones finish (the
    // hardware dispatcher is the work queue); each XCD takes runs of
    // kItemRun consecutive (segment, group) items, the NG groups of a
    // segment adjacent, so neighbouring nodes and the groups of one segment
    // share that XCD's L2
    __shared__ MixItemLds<MT> sh;
    const int nitem = a.nbatch * a.nseg * NG;
    const int it = item_of_block();
    if (it < nitem)
        mix_item_run<MT, NG>(a, it, sh);
}

}  // namespace

template <int M>
void launch_mix_item(hipStream_t s, dim3 grid, const CalcArgs& a, int ng)
{
    constexpr int lo = item_groups_lo(M);
    if (ng == item_groups_many(M))
        hipLaunchKernelGGL((gram_mixed_item_kernel<M, item_groups_many(M)>), grid, dim3(64), 0, s, a);
    else if (ng == lo + 1)
        hipLaunchKernelGGL((gram_mixed_item_kernel<M, lo + 1>), grid, dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL((gram_mixed_item_kernel<M, lo>), grid, dim3(64), 0, s, a);
}

hipError_t launch_gram_mixed(hipStream_t s, const CalcArgs& a)
{
    const int MT = (a.m + 15) / 16;
    if (a.nbatch == 0)
        return hipSuccess;
    if (MT >= 1 && MT <= 10) {
        // tile groups per segment: one of the two candidates of this MT (the
        // smaller by default)
        const int lo = item_groups_lo(MT);
        const long long nlist = (long long)a.nbatch * a.nseg;
        const int ng = few_lists(MT, nlist) ? item_groups_many(MT) : (a.tile_groups == lo + 1 ? lo + 1 : lo);
        const long long nitem = (long long)a.nbatch * a.nseg * ng;
        const dim3 igrid(item_grid(nitem));
        switch (MT) {
        case 1: launch_mix_item<1>(s, igrid, a, ng); break;
        case 2: launch_mix_item<2>(s, igrid, a, ng); break;
        case 3: launch_mix_item<3>(s, igrid, a, ng); break;
        case 4: launch_mix_item<4>(s, igrid, a, ng); break;
        case 5: launch_mix_item<5>(s, igrid, a, ng); break;
        case 6: launch_mix_item<6>(s, igrid, a, ng); break;
        case 7: launch_mix_item<7>(s, igrid, a, ng); break;
        case 8: launch_mix_item<8>(s, igrid, a, ng); break;
        case 9: launch_mix_item<9>(s, igrid, a, ng); break;
        default: launch_mix_item<10>(s, igrid, a, ng); break;
        }
        return hipGetLastError();
    }
    return hipErrorInvalidValue;   // m > 160 is refused at configuration
}

}  // namespace enkfg
