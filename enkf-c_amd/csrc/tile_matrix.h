// tile_matrix.h -- symmetric matrices of up to 160 x 160 in the registers of
// one wavefront, as 16 x 16 FP64 tiles in the accumulator layout of
// v_mfma_f64_16x16x4_f64: register r of lane l holds element
// (4 r + l / 16, l % 16).
//
// In that layout register r is at once the B operand of k-step r (rows 4 r ..
// 4 r + 3 of the tile) and the A operand of k-step r of the tile's transpose.
// So X^T Y of two tiles takes four MFMA instructions and no data movement,
// and everything below is written in products of that form.
#pragma once

#include <type_traits>

#include "enkfg_internal.h"
#include "gram_layout.h"

namespace enkfg {

typedef double tile4 __attribute__((ext_vector_type(4)));

// f(integral_constant B), ..., f(integral_constant E - 1): loops whose tile
// indices are constants whatever the unroller decides (a tile indexed at run
// time would put them all in scratch memory)
template <int B, int E, class F>
__device__ __attribute__((always_inline)) inline void static_for(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// 1/d for a pivot d >= 1 (the pivots of I + S^T S are Schur complements of
// at least 1): the hardware estimate refined by two Newton-Raphson steps
// r <- r + r (1 - d r), within an ulp of 1/d
__device__ inline double recip_pivot(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    double e = fma(-d, r, 1.0);
    r = fma(r, e, r);
    e = fma(-d, r, 1.0);
    return fma(r, e, r);
}

// acc += X^T Y
__device__ __attribute__((always_inline)) inline void tile_mma(tile4& acc, const tile4& x, const tile4& y)
{
#pragma unroll
    for (int r = 0; r < 4; ++r)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[r], y[r], acc, 0, 0, 0);
}

// the tile as it is at this point of the program: without this the compiler
// moves the end of its computation down to its use and keeps the operands
__device__ __attribute__((always_inline)) inline void tile_pin(tile4& x) { asm volatile("" : "+v"(x)); }

// lane K of each row of 16 lanes, in every lane of the row
template <int K>
__device__ __attribute__((always_inline)) inline double row_bcast(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = (int)(unsigned)b, hi = (int)(unsigned)(b >> 32);
    const unsigned l = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, 0x150 | K, 0xf, 0xf, true);
    const unsigned h = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, 0x150 | K, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)h << 32) | l);
}

// the 16 lanes of row G, in every row of 16 lanes: the halves swapped against
// a copy give either half in both, then the rows likewise
template <int G>
__device__ __attribute__((always_inline)) inline unsigned rows_bcast32(unsigned v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const unsigned h = (G >> 1) ? a[1] : a[0];
    const auto b = __builtin_amdgcn_permlane16_swap(h, h, false, false);
    return (G & 1) ? b[1] : b[0];
#else
    return v;
#endif
}

template <int G>
__device__ __attribute__((always_inline)) inline double rows_bcast(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned l = rows_bcast32<G>((unsigned)b), h = rows_bcast32<G>((unsigned)(b >> 32));
    return __builtin_bit_cast(double, ((unsigned long long)h << 32) | l);
}

// Pivot K of the symmetric sweep on one tile: A_ij -= A_iK A_Kj / d for i, j
// != K, A_iK = A_iK / d, A_Kj = A_Kj / d, A_KK = -1 / d.  One multiply-add
// per register: lanes of column K start from 0 with the factor -1/d, those of
// row K from 0 with u = -1.
template <int K>
__device__ __attribute__((always_inline)) inline void sweep_pivot(tile4& x, int col, int grp, bool& bad, double& det)
{
    constexpr int RK = K >> 2, GK = K & 3;
    const double p = rows_bcast<GK>(x[RK]);   // A_K,col
    const double d = row_bcast<K>(p);
    bad |= !(d > 0.0);
    det *= d;
    const double pinv = recip_pivot(d);
    const bool kc = col == K, kr = grp == GK;
    const double ws = kc ? -pinv : p * pinv;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        double u = row_bcast<K>(x[r]);         // A_row,K
        double v = kc ? 0.0 : x[r];
        if (r == RK) {
            v = kr ? 0.0 : v;
            u = kr ? -1.0 : u;
        }
        x[r] = fma(-u, ws, v);
    }
    if constexpr (K < 15)
        sweep_pivot<K + 1>(x, col, grp, bad, det);
}

// x <- -x^-1 for a symmetric positive definite tile; det is its determinant
__device__ __attribute__((always_inline)) inline void tile_sweep(tile4& x, int lane, bool& bad, double& det)
{
    det = 1.0;
    sweep_pivot<0>(x, lane & 15, lane >> 4, bad, det);
}

// index of tile (i, j), i <= j, in the upper triangle stored row by row
template <int MT>
__host__ __device__ constexpr int tri_at(int i, int j)
{
    return i * MT - i * (i - 1) / 2 + (j - i);
}

// Block elimination of the matrix in x (upper tiles, row by row), in place:
// with D_k the inverse of the k-th diagonal Schur complement and U_kj = D_k
// A_kj the rows of the unit upper block factor (A = U^T diag(D^-1) U), tile
// (k, k) becomes -D_k and tile (k, j) becomes -U_kj.
//
//   -U_kj = (-D_k)^T A_kj;   A_ij += (-U_ki)^T A_kj,  k < i <= j
template <int MT>
__device__ __attribute__((always_inline)) inline void tile_eliminate(tile4* x, int lane, bool& bad, double& logdet)
{
    double mant = 1.0;
    int ex = 0;
    static_for<0, MT>([&](auto kc) {
        constexpr int k = kc;
        double det;
        tile_sweep(x[tri_at<MT>(k, k)], lane, bad, det);
        int e;
        mant = frexp(mant * det, &e);
        ex += e;
        static_for<k + 1, MT>([&](auto jc) {
            constexpr int j = jc;
            tile4 u = {0.0, 0.0, 0.0, 0.0};
            tile_mma(u, x[tri_at<MT>(k, k)], x[tri_at<MT>(k, j)]);
            static_for<k + 1, j>([&](auto ic) {
                constexpr int i = ic;
                tile_mma(x[tri_at<MT>(i, j)], x[tri_at<MT>(k, i)], x[tri_at<MT>(k, j)]);
            });
            tile_mma(x[tri_at<MT>(j, j)], u, x[tri_at<MT>(k, j)]);
            x[tri_at<MT>(k, j)] = u;
        });
    });
    logdet = log(mant) + (double)ex * 0.69314718055994530942;
}

// After tile_eliminate: tile (i, j), i < j, becomes V_ji, V = U^-T the unit
// lower block factor of the inverse (A^-1 = V^T diag(D) V):
//   V_ji = (-U_ij)^T + sum_{i < l < j} (-U_lj)^T V_li
// Row i of the tiles is column i of V, and needs rows >= i only, so it is
// done in place.
template <int MT>
__device__ __attribute__((always_inline)) inline void tile_invert_factor(tile4* x, int lane)
{
    tile4 eye;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        eye[r] = (4 * r + (lane >> 4) == (lane & 15)) ? 1.0 : 0.0;
    static_for<0, MT>([&](auto ic) {
        constexpr int i = ic;
        static_for<i + 1, MT>([&](auto jc) {
            constexpr int j = jc;
            tile4 v = {0.0, 0.0, 0.0, 0.0};
            tile_mma(v, x[tri_at<MT>(i, j)], eye);
            static_for<i + 1, j>([&](auto lc) {
                constexpr int l = lc;
                tile_mma(v, x[tri_at<MT>(l, j)], x[tri_at<MT>(i, l)]);
            });
            x[tri_at<MT>(i, j)] = v;
        });
    });
}

// wavefronts per SIMD that the tiles' registers allow (8 per tile, and about
// 60 beside them)
__host__ __device__ constexpr int tile_waves(int MT) { return MT <= 3 ? 4 : (MT <= 6 ? 2 : 1); }

}  // namespace enkfg
