// gram_layout.h -- tile enumeration of the Gram kernels and the layout of the
// Gram scratch that the factor kernel reads.
#pragma once

#include <stddef.h>

#include "enkfg_internal.h"

namespace enkfg {

// Upper-triangular 16x16 tiles (I <= J) of an MT x MT tile grid, enumerated
// row by row
__host__ __device__ constexpr int tri_count(int MT) { return MT * (MT + 1) / 2; }

// The item Gram kernels split a segment's tri_count(MT) tiles into NG groups
// (group g: tiles g, g + NG, ...), one wavefront each; the two candidates per MT
// are lo and lo + 1.  An observation is read and converted once per group, so
// fewer groups do less work, as far as a group's accumulators and operands
// fit the 256 registers of a lane beside two wavefronts a SIMD.  m = 96: all
// 21 tiles in one wavefront take 244 registers (mixed 217); FP64 calc on the
// 51x1500x1800 tile 379 ms against 412 for two groups of unpipelined k-steps.
// Up to m = 64 a segment has ten tiles or fewer and two wavefronts are kept,
// for launches of few nodes.  From MT = 7 on the counts (3, 4, 4, 5) are those
// that were measured with the kernels before the pipelined k-steps (156 to 193
// registers, mixed 180 to 228); 2, 2, 3 and 4 would fit too, with 193, 234, 215
// and 214 registers (mixed 205, 238, 230, 247) and no vector spills, and have
// not been measured.
__host__ __device__ constexpr int item_groups_lo(int MT)
{
    return MT <= 4 ? 2 : (MT <= 6 ? 1 : (MT == 7 ? 3 : (MT <= 9 ? 4 : 5)));
}

// Launches of few nodes: about three tiles a wavefront, so that a list's
// chunks take less time each and more wavefronts share the work (9 nodes of
// four lists, the longest 3,000 obs, m = 96: 0.41 ms with two groups).  Used
// where even then the items are fewer than kManyItems, two wavefronts per
// SIMD (few_lists), whatever CalcArgs::tile_groups asks for; such launches are
// not tuned.  The matrices are the same bit for bit.
__host__ __device__ constexpr int item_groups_many(int MT) { return MT <= 4 ? item_groups_lo(MT) + 1 : (tri_count(MT) + 2) / 3; }
constexpr long long kManyItems = 2048;
inline bool few_lists(int MT, long long nlist) { return nlist * item_groups_many(MT) <= kManyItems; }

// The items (segment, tile group) of the item Gram kernels are dealt to the 8
// XCDs in runs of kItemRun.  Block i runs on XCD i % 8 (the hardware
// dispatcher deals blocks round-robin), and XCD x takes runs x, x + 8,
// x + 16, ...  A run of 64 items (8 nodes at 2 groups and 4 obstypes) keeps
// neighbouring nodes, whose lists share rows, on one L2, while the runs
// spread each XCD's share over the whole batch.  Contiguous eighths of the
// batch leave the XCD with the heaviest nodes finishing last (FP64 calc on
// the 51x1500x1800 tile: 683 ms, against 667 ms with runs of 16 to 128 items
// and 734 ms with single items).
constexpr int kItemRun = 64;

__device__ inline int item_of_block()
{
    const int x = (int)(blockIdx.x % 8), j = (int)(blockIdx.x / 8);
    return ((j / kItemRun) * 8 + x) * kItemRun + j % kItemRun;
}

// Item `it` of an item Gram launch with NG tile groups per segment: node
// slot bn of the batch, segment seg, group g.  Items run segment by segment
// in the order a.seg_order (obstypes by decreasing total list length), the
// batch's nodes in order within a segment and the NG groups of a (node,
// segment) adjacent.  So the longest items start first and a launch ends on
// short ones: with the nodes' four segments interleaved, the last few of the
// longest items ran alone at the end of each launch (in a copy of the chunk
// loop with 231, 116, 20 and 20 chunks per segment, 47 against 64 TFLOP/s
// for uniform items).  Within a run of kItemRun items the nodes are
// neighbours with lists of one obstype, which share rows in L2.
struct ItemRef {
    int bn, seg, g;
};

__device__ inline ItemRef item_ref(const CalcArgs& a, int it, int NG)
{
    const int per = a.nbatch * NG;
    const int sr = it / per;
    const int rem = it - sr * per;
    ItemRef r;
    r.bn = rem / NG;
    r.g = rem - r.bn * NG;
    r.seg = a.seg_order ? a.seg_order[sr] : sr;
    return r;
}

// blocks of an item Gram launch: a whole number of rounds of 8 runs, over
// which item_of_block is one to one
inline unsigned item_grid(long long nitem)
{
    const long long round = 8LL * kItemRun;
    return (unsigned)(round * ((nitem + round - 1) / round));
}
__host__ __device__ constexpr int tri_I(int MT, int f)
{
    int I = 0;
    while (f >= MT - I) {
        f -= MT - I;
        ++I;
    }
    return I;
}
__host__ __device__ constexpr int tri_J(int MT, int f)
{
    int I = 0;
    while (f >= MT - I) {
        f -= MT - I;
        ++I;
    }
    return I + f;
}

// The Gram scratch of one (node, segment): the upper-triangle tiles in the
// order above, each 16 x 16 row-major.  Row-major is the accumulator layout of
// v_mfma_f64_16x16x4_f64 with lane l's register i at 64 i + l, so the Gram
// kernel stores and the factor kernels load whole 512-byte runs (and 21
// tiles instead of 36 for m = 96).
__host__ __device__ constexpr size_t gram_size(int MT) { return (size_t)tri_count(MT) * 256; }

}  // namespace enkfg
