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

// 1/d for d > 0 (the pivots of I + S^T S are Schur complements of at least
// 1): the hardware estimate refined by two Newton-Raphson steps
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

// a zero tile that the compiler forms only here, in program order: products
// into it are not taken ahead of the outputs of earlier tiles, for which
// there are no registers
__device__ __attribute__((always_inline)) inline tile4 ordered_zero()
{
    double z = 0.0;
    asm volatile("" : "+v"(z)::"memory");
    return tile4{z, z, z, z};
}

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

// Pivot K of the elimination of one symmetric tile x, with its column
// operations collected in f: x_ij -= x_iK x_Kj / d and f_ij -= f_iK x_Kj / d for
// j > K.  Rows of x above and of f below K do not matter any more, or yet;
// dcol receives the pivot in the lanes of column K.
template <int K>
__device__ __attribute__((always_inline)) inline void chol_pivot(tile4& x, tile4& f, double& dcol, int col, bool& bad)
{
    constexpr int RK = K >> 2, GK = K & 3;
    const double p = rows_bcast<GK>(x[RK]);   // x_K,col
    const double d = row_bcast<K>(p);
    bad |= !(d > 0.0);
    dcol = col == K ? d : dcol;
    if constexpr (K < 15) {
        const double ws = col > K ? p * recip_pivot(d) : 0.0;
#pragma unroll
        for (int r = RK; r < 4; ++r)
            x[r] = fma(-row_bcast<K>(x[r]), ws, x[r]);
#pragma unroll
        for (int r = 0; r <= RK; ++r)
            f[r] = fma(-row_bcast<K>(f[r]), ws, f[r]);
        chol_pivot<K + 1>(x, f, dcol, col, bad);
    }
}

// 1/sqrt(d): the hardware estimate and two Newton-Raphson steps
__device__ inline double rsqrt_pivot(double d)
{
    double y = __builtin_amdgcn_rsq(d);
    double e = fma(-d * y, y, 1.0);
    y = fma(0.5 * y, e, y);
    e = fma(-d * y, y, 1.0);
    return fma(0.5 * y, e, y);
}

// x <- W, upper triangular, W W^T = x^-1, for a symmetric positive definite
// tile (x = R^T R, W = R^-1); the lanes of column k add log2 of pivot k to ld
__device__ __attribute__((always_inline)) inline void tile_chol(tile4& x, int lane, bool& bad, float& ld)
{
    tile4 f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        f[r] = (4 * r + (lane >> 4) == (lane & 15)) ? 1.0 : 0.0;
    double dcol = 1.0;
    chol_pivot<0>(x, f, dcol, lane & 15, bad);
    ld += __builtin_amdgcn_logf((float)__builtin_amdgcn_frexp_mant(dcol)) + (float)__builtin_amdgcn_frexp_exp(dcol);
    const double s = rsqrt_pivot(dcol);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        x[r] = f[r] * s;
}

// index of tile (i, j), i <= j, in the upper triangle stored row by row
template <int MT>
__host__ __device__ constexpr int tri_at(int i, int j)
{
    return i * MT - i * (i - 1) / 2 + (j - i);
}

// Block Cholesky factorisation A = R^T R of the matrix in x (upper tiles, row
// by row), in place: tile (k, k) becomes W_k = R_kk^-1 and tile (k, j) becomes
// -R_kj.
//
//   R_kj = W_k^T A_kj;   A_ij += (-R_ki)^T R_kj,  k < i <= j
//
// log2det: log2 of the determinant, in single precision: the sum of the
// pivots' (their product leaves the range of a double where 16 of them exceed
// 1e19).
//
// With the inverse of a triangular diagonal block the error stays within
// cond(R_kk) of the unblocked elimination's; with the inverse of the block
// itself (cond(R_kk)^2) w lost two digits on 96 + 48 members with clustered
// obs (3e-10 of max |w| against the oracle).
template <int MT>
__device__ __attribute__((always_inline)) inline void tile_eliminate(tile4* x, int lane, bool& bad, float& log2det)
{
    float ld = 0.0f;
    auto factor = [&](tile4& d) {
        int ln = lane;
        asm volatile("" : "+v"(ln));   // (the pivots' masks are not kept between them)
        tile_chol(d, ln, bad, ld);
    };
    auto eliminate = [&](auto kc, const tile4& d) {
        constexpr int k = kc;
        x[tri_at<MT>(k, k)] = d;
        static_for<k + 1, MT>([&](auto jc) {
            constexpr int j = jc;
            tile4 u = {0.0, 0.0, 0.0, 0.0};
            tile_mma(u, d, x[tri_at<MT>(k, j)]);
            const tile4 n = -u;
            static_for<k + 1, j>([&](auto ic) {
                constexpr int i = ic;
                tile_mma(x[tri_at<MT>(i, j)], x[tri_at<MT>(k, i)], u);
            });
            tile_mma(x[tri_at<MT>(j, j)], n, u);
            x[tri_at<MT>(k, j)] = n;
        });
    };
    if constexpr (MT <= 3) {
        static_for<0, MT>([&](auto kc) {
            tile4 d = x[tri_at<MT>(kc, kc)];
            factor(d);
            eliminate(kc, d);
        });
    } else {
        // One copy of the diagonal factor's code for all k: unrolled, it was
        // most of the kernels' 40 to 130 KB and did not stay in the
        // instruction cache (ETKF, 4,050 nodes, m = 96: 7.1 -> 4.3 ms; for m =
        // 24 the choice of the tile costs more, 0.32 against 0.22 ms)
#pragma unroll 1
        for (int k = 0; k < MT; ++k) {
            // (the asm keeps the cases apart: merged, they would index the
            // tiles at run time, in scratch memory)
            tile4 d = {0.0, 0.0, 0.0, 0.0};
            static_for<0, MT>([&](auto kc) {
                constexpr int kk = kc;
                if (k == kk) {
                    d = x[tri_at<MT>(kk, kk)];
                    asm volatile("" : "+v"(d) : "n"(kk));
                }
            });
            factor(d);
            static_for<0, MT>([&](auto kc) {
                constexpr int kk = kc;
                if (k == kk) {
                    asm volatile("" : "+v"(d) : "n"(kk));
                    eliminate(kc, d);
                }
            });
        }
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1)
        ld += __shfl_xor(ld, o);
    log2det = ld;
}

// After tile_eliminate: tile (i, j), i <= j, becomes V_ji of the lower
// triangular V = R^-T (A^-1 = V^T V):
//   V_ii = W_i^T;   V_ji = W_j^T sum_{i <= l < j} (-R_lj)^T V_li
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
        tile4 d = {0.0, 0.0, 0.0, 0.0};
        tile_mma(d, x[tri_at<MT>(i, i)], eye);
        x[tri_at<MT>(i, i)] = d;
        static_for<i + 1, MT>([&](auto jc) {
            constexpr int j = jc;
            tile4 t = {0.0, 0.0, 0.0, 0.0}, v = {0.0, 0.0, 0.0, 0.0};
            static_for<i, j>([&](auto lc) {
                constexpr int l = lc;
                tile_mma(t, x[tri_at<MT>(l, j)], x[tri_at<MT>(i, l)]);
            });
            tile_mma(v, x[tri_at<MT>(j, j)], t);
            x[tri_at<MT>(i, j)] = v;
        });
    });
}

// After tile_invert_factor: f(i, j, tile) for the tiles (i, j), i <= j, of the
// inverse, sum_{l >= j} V_li^T V_lj, one after another
template <int MT, class F>
__device__ __attribute__((always_inline)) inline void tile_inverse(const tile4* x, F&& f)
{
    static_for<0, MT>([&](auto jc) {
        constexpr int j = jc;
        static_for<0, j + 1>([&](auto ic) {
            constexpr int i = ic;
            tile4 v = ordered_zero();
            static_for<j, MT>([&](auto lc) {
                constexpr int l = lc;
                tile_mma(v, x[tri_at<MT>(i, l)], x[tri_at<MT>(j, l)]);
            });
            tile_pin(v);
            f(ic, jc, v);
        });
    });
}

// wavefronts per SIMD for which the kernels are compiled: a lane's share of a
// SIMD's 512 registers is 8 for each tile and what the kernel needs beside
// them, which is more than the rest of the share for some MT: the DEnKF and
// trace kernels spill 10 and 8 registers at MT = 6, 14 and 8 at 8, 206 and 130
// at 9, 789 and 542 at 10, the ETKF kernel 22, 99, 44, 24, 34, 304 and 780 at
// 2, 3, 6, 7, 8, 9 and 10 (compiler's report).  Other counts for these have
// not been measured.
__host__ __device__ constexpr int tile_waves(int MT) { return MT <= 3 ? 4 : (MT <= 6 ? 2 : 1); }

constexpr double kDfsMin = 1.0e-6;   // DFS_MIN, calc/transforms.c:32

__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
        v += __shfl_xor(v, o);
    return v;
}

// The upper tiles stored at g, a tile at a time in the accumulator layout.  Of
// a diagonal tile the upper triangle is read for both: its two triangles
// differ by their rounding (in the mixed Gram by that of FP32 sums), and the
// elimination takes the matrix as symmetric.
template <int MT, int F0, int N>
__device__ __attribute__((always_inline)) inline void read_tiles(const double* g, int lane, tile4* t)
{
    int sym[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + (lane >> 4), col = lane & 15;
        sym[r] = row <= col ? 16 * row + col : 16 * col + row;
    }
    static_for<F0, F0 + N>([&](auto fc) {
        constexpr int f = fc;
        constexpr bool diag = tri_I(MT, f) == tri_J(MT, f);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            t[f - F0][r] = g[(size_t)f * 256 + (diag ? sym[r] : 64 * r + lane)];
    });
}

// x <- I + the Gram matrices of segments s0 .. s1 - 1 (ONE: s0) of batch node bnode;
// returns the trace of the Gram matrix G (NORM2: norm2 <- |G|^2)
template <int MT, bool ONE, bool NORM2 = false>
__device__ __attribute__((always_inline)) inline double load_tiles(const CalcArgs& a, int bnode, int node, int s0,
                                                                   int s1, int lane, tile4* x, double* norm2 = nullptr)
{
    constexpr int NT = tri_count(MT);
    // the first segment's tiles are loaded straight into x, all at once; the
    // others' kGroup at a time (the loads in flight need registers beside x)
    constexpr int kGroup = MT <= 7 ? 7 : 4;
    const double* g = a.gram + ((size_t)bnode * a.nseg + s0) * gram_size(MT);
    int s = s0;
    if (!ONE && a.pertype)
        while (s < s1 - 1 && a.counts[(size_t)node * a.ntypes + s] == 0)
            ++s;
    const double* gs = g + (size_t)(s - s0) * gram_size(MT);
    read_tiles<MT, 0, NT>(gs, lane, x);
#pragma unroll
    for (int f = 0; f < NT; ++f)
        tile_pin(x[f]);
    __builtin_amdgcn_sched_barrier(0);
    for (++s; !ONE && s < s1; ++s) {
        if (a.pertype && a.counts[(size_t)node * a.ntypes + s] == 0)
            continue;
        gs = g + (size_t)(s - s0) * gram_size(MT);
        static_for<0, (NT + kGroup - 1) / kGroup>([&](auto gc) {
            constexpr int f0 = gc * kGroup;
            constexpr int n = f0 + kGroup < NT ? kGroup : NT - f0;
            tile4 t[n];
            read_tiles<MT, f0, n>(gs, lane, t);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < n; ++f)
                x[f0 + f] += t[f];
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    if (!ONE) {
#pragma unroll
        for (int f = 0; f < NT; ++f)
            tile_pin(x[f]);
    }
    if constexpr (NORM2) {
        double d = 0.0, o = 0.0;   // of the diagonal tiles, and of the others
        static_for<0, NT>([&](auto fc) {
            constexpr int f = fc;
            double& v = tri_I(MT, f) == tri_J(MT, f) ? d : o;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v = fma(x[f][r], x[f][r], v);
        });
        *norm2 = wave_sum(d + 2.0 * o);
    }
    double tr = 0.0;
#pragma unroll
    for (int k = 0; k < MT; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * r + (lane >> 4) == (lane & 15)) {
                tr += x[tri_at<MT>(k, k)][r];
                x[tri_at<MT>(k, k)][r] += 1.0;
            }
    return wave_sum(tr);
}

template <int MT>
struct TileLds {
    double b[16 * MT];      // S^T s over the node's segments
    double g[16 * MT];      // adjoint: dJ/dw of the node
    double t[16][17];       // a tile, for its transpose
};

}  // namespace enkfg
