// loc_kernels.hip -- GPU localisation: for every node of the stride grid, the
// list of (obs, taper coefficient) that obs_findlocal
// (common/observations.c:1837-1927) returns.
//
// Two searches give the same lists.
//
// The box search (loc_box_kernel) is what the calc uses, which needs the
// lists in no particular order.  Rows (and so S) are sorted along a Morton
// curve per type; 64 consecutive rows make a leaf, 64 boxes a box of the next
// level, three levels in all.  One wavefront takes one (node, obstype): a
// step tests 64 boxes or 64 observations with coalesced loads.  Distances
// and tapers use the reference's operation order in IEEE double with no
// contraction, and a box is skipped only when its distance, rounded in the
// same order, exceeds the radius -- rounding is monotone, so no observation
// of it can be within the radius -- so the set and the taper bits are the
// tree search's.  By the same argument the tree search reaches every
// observation within the radius whose distance along each axis is below the
// radius.  One at exactly the radius along an axis may lie behind a split
// that was pruned: where counting finds any, it is done again with the trees,
// and these observations climb theirs (walk_reaches).  A non-finite second
// coordinate is in no list, in the tree on no finite observation's far side,
// and left out of the boxes' bounds.
//
// The tree search walks the reference's own kd-trees (sequential insertion,
// obs_createkdtrees) in the preorder of _kd_findnodeswithinrange
// (common/kdtree.c:516-540) -- node, then the child on the query's side (left
// iff dx <= 0), then the other child iff |dx| < range -- without a stack by
// following parent links: on the way up, a node is re-examined to decide
// whether the far child is still to be visited, which depends only on that
// node and the query.  Its lists are in the reference's order, element for
// element: enkfg_localise and enkfg_get_localobs return those.  It also
// serves NLOBSMAX, which keeps candidates at equal distance in visiting order.
//
// What bounds them, on the 51x1500x1800 tile (300,000 nodes, four types,
// 1.86G entries, 22 GB of lists): the tree walk by the traffic of its node
// loads beyond L2 and by the depth of the trees (walking and compacting the
// lists took 100 ms with the observations in random order, 991 ms in
// enkf_prep order); the box search, counting and filling, by FP64 issue (a
// leaf's distances twice, the tapers once) at 17.5 ms in either order.  On
// 200 x 240 cells and 9 nodes it takes 0.14 ms against 13 ms: a walk's
// dependent loads are one chain per thread, a box search's steps load 64
// boxes or 256 observations each.
//
// The obs indices in the lists are device rows; the host maps them back to
// observation indices.
#include <algorithm>

#include "enkfg_internal.h"

namespace enkfg {

namespace {

constexpr int kStatusOK = 0;

__device__ inline double taper_gc(double x)
{
    // common/utils.c:1425-1443
    if (x >= 1.0)
        return 0.0;
    x *= 2.0;
    double x2 = x * x;
    double x3 = x2 * x;
    double f;
    if (x < 1.0)
        f = 1.0 + x2 * (-x3 / 4.0 + x2 / 2.0) + x3 * (5.0 / 8.0) - x2 * (5.0 / 3.0);
    else
        f = x2 * (x3 / 12.0 - x2 / 2.0) + x3 * (5.0 / 8.0) + x2 * (5.0 / 3.0) - x * 5.0 + 4.0 - (2.0 / 3.0) / x;
    return (f >= 0.0) ? f : 0.0;
}

__device__ inline double calclcoeff(const TypeInfo& t, double dist)
{
    // common/obstypes.c:800-810
    double sum = 0.0;
    for (int i = 0; i < t.nlocrad; ++i)
        if (dist <= t.locrad[i])
            sum += t.locweight[i] * taper_gc(dist / t.locrad[i]);
    return sum;
}

// Depth-first range search over one tree; calls emit(node, distsq) for every
// hit in the reference's visiting order.  The split dimension is the depth
// modulo ND, tracked on the way down and up.  Each step selects the next
// node without branching (down to the near child if there is one, else to
// the far child if the range crosses the split, else up; coming up from the
// near child, to the far child under the same condition, else further up),
// so that the lanes of a wave at different stages of their walks stay in
// one instruction stream.
template <int ND, class Emit>
__device__ inline void range_walk_nd(const KdNode* __restrict__ tree, const double* q, double range, Emit&& emit)
{
    const double r2 = range * range;
    const double q0 = q[0], q1 = q[1], q2 = ND == 3 ? q[2] : 0.0;
    int node = 0;
    int from = -1;
    int dir = 0;
    bool down = true;

    while (node >= 0) {
        const KdNode nd = tree[node];
        const double cd = dir == 0 ? nd.x : ((ND == 2 || dir == 1) ? nd.y : nd.z);
        const double qd = dir == 0 ? q0 : ((ND == 2 || dir == 1) ? q1 : q2);
        const double dx = qd - cd;
        if (down) {
            // kd_findnodeswithinrange's sum, in its order (kdtree.c:529-533)
            double distsq = 0.0;
            double d = nd.x - q0;
            distsq += d * d;
            d = nd.y - q1;
            distsq += d * d;
            if (ND == 3) {
                d = nd.z - q2;
                distsq += d * d;
            }
            if (distsq <= r2)
                emit(node, distsq);
        }
        const int left = (nd.link & 0x80000000u) ? node + 1 : -1;
        const bool lside = dx <= 0.0;
        const int near = lside ? left : nd.right;
        const int far = lside ? nd.right : left;
        const int parent = (int)(nd.link & 0x7fffffffu) - 1;
        const bool farok = fabs(dx) < range && far >= 0;
        const bool tonear = down && near >= 0;
        const bool tofar = !tonear && farok && (down || from == near);
        const bool ndown = tonear || tofar;
        from = node;
        node = tonear ? near : (tofar ? far : parent);
        dir = ndown ? (dir + 1 == ND ? 0 : dir + 1) : (dir == 0 ? ND - 1 : dir - 1);
        down = ndown;
    }
}

template <class Emit>
__device__ inline void range_walk(const KdNode* __restrict__ tree, int ndim, const double* q, double range, Emit&& emit)
{
    if (ndim == 3)
        range_walk_nd<3>(tree, q, range, emit);
    else
        range_walk_nd<2>(tree, q, range, emit);
}

// Thread mapping: one thread per (node, obstype); a wave takes an 8 x 8 tile
// of the stride grid and one obstype, so its lanes walk nearly the same
// paths of one tree and their node loads coalesce.  ni is the grid's row
// length (nnode = ni nj); tiles are row-major within a type.
// consecutive walk items per XCD run: four 8 x 8 blocks of tiles (runs of
// one block: localisation 103-105 ms on the tile, of four 101-102 ms, of
// sixteen 135 ms: the XCDs with the densest regions then finish last)
constexpr int kWalkRun = 256;

__device__ inline bool thread_node(int nnode, int ni, int ntypes, int& t, int& node)
{
    const int nj = nnode / ni;
    const int ti = (ni + 7) / 8, tj = (nj + 7) / 8;
    const int sti = (ti + 7) / 8, stj = (tj + 7) / 8;   // 8 x 8 blocks of tiles
    const long long per_type = (long long)sti * stj * 64 * 64;
    // Tiles are ordered in 8 x 8 blocks of tiles (64 x 64 nodes), row-major
    // within and between blocks.  Blocks go to the 8 XCDs round-robin; each
    // XCD takes runs of kWalkRun consecutive (type, tile) items -- four
    // blocks of tiles -- so the walks in flight on one L2 cover a compact patch of
    // the grid, and the runs are dealt round-robin, so dense and sparse
    // regions spread over all XCDs (walk_grid rounds the grid up to a
    // multiple of 8 runs; items past the grid's edge return)
    const unsigned s = blockIdx.x / 8, x = blockIdx.x % 8;
    const long long item = ((long long)(s / kWalkRun) * 8 + x) * kWalkRun + s % kWalkRun;
    const long long gid = item * blockDim.x + threadIdx.x;
    if (gid >= per_type * ntypes)
        return false;
    t = (int)(gid / per_type);
    const long long rem = gid - (long long)t * per_type;
    const int tile = (int)(rem / 64), lane = (int)(rem % 64);
    const int sb = tile / 64, wi = tile % 64;
    const int tx = (sb % sti) * 8 + wi % 8, ty = (sb / sti) * 8 + wi / 8;
    if (tx >= ti || ty >= tj)
        return false;
    const int i = tx * 8 + lane % 8, j = ty * 8 + lane / 8;
    if (i >= ni || j >= nj)
        return false;
    node = j * ni + i;
    return true;
}

__global__ void __launch_bounds__(64) loc_count_kernel(int nnode, int ni, const double* __restrict__ qxyz,
                                                        const unsigned char* __restrict__ isglobal,
                                                        const unsigned char* __restrict__ visible,
                                                        const KdNode* __restrict__ nodes,
                                                        const int* __restrict__ noderow,
                                                        const TypeInfo* __restrict__ types, int ntypes,
                                                        const short* __restrict__ status, int* __restrict__ counts,
                                                        int* __restrict__ raw)
{
    int t, node;
    if (!thread_node(nnode, ni, ntypes, t, node))
        return;
    double q[3] = {qxyz[3 * (size_t)node], qxyz[3 * (size_t)node + 1], qxyz[3 * (size_t)node + 2]};
    const bool glob = isglobal[node] != 0;
    const TypeInfo& ti = types[t];
    int n = 0, nraw = 0;
    if (ti.searchable && (visible == nullptr || visible[t])) {
        if (glob) {
            n = ti.nids;   // obs_getglobal: all obs of the type, no status check
        } else if (ti.nnode > 0 && ti.nlobsmax != ENKFG_NLOBSMAX_NONE) {
            // NLOBSMAX: every hit is a candidate; the sort kernel selects
            range_walk(nodes + ti.node0, ti.ndim, q, ti.range, [&](int, double) { nraw++; });
        } else if (ti.nnode > 0) {
            range_walk(nodes + ti.node0, ti.ndim, q, ti.range, [&](int v, double) {
                if (status[noderow[ti.node0 + v]] == kStatusOK)
                    n++;
            });
        }
    }
    counts[(size_t)node * ntypes + t] = n;
    if (raw != nullptr)
        raw[(size_t)node * ntypes + t] = nraw;
}

// NLOBSMAX candidates of a (node, type): rows and squared distances in the
// reference's visiting order
__global__ void __launch_bounds__(64) loc_rawfill_kernel(int nnode, int ni, const double* __restrict__ qxyz,
                                                         const unsigned char* __restrict__ isglobal,
                                                         const unsigned char* __restrict__ visible,
                                                         const KdNode* __restrict__ nodes,
                                                         const int* __restrict__ noderow,
                                                         const TypeInfo* __restrict__ types, int ntypes,
                                                         const long long* __restrict__ rawoff, int* __restrict__ rrow,
                                                         double* __restrict__ rd2)
{
    int t, node;
    if (!thread_node(nnode, ni, ntypes, t, node))
        return;
    const TypeInfo& ti = types[t];
    if (isglobal[node] || !ti.searchable || !(visible == nullptr || visible[t]) || ti.nnode == 0 ||
        ti.nlobsmax == ENKFG_NLOBSMAX_NONE)
        return;
    double q[3] = {qxyz[3 * (size_t)node], qxyz[3 * (size_t)node + 1], qxyz[3 * (size_t)node + 2]};
    long long o = rawoff[(size_t)node * ntypes + t];
    range_walk(nodes + ti.node0, ti.ndim, q, ti.range, [&](int v, double distsq) {
        rrow[o] = noderow[ti.node0 + v];
        rd2[o] = distsq;
        o++;
    });
}

// The candidates of one (node, type) sorted by distance, ties in visiting
// order (the stable sort of kd_findnodeswithinrange's qsort on this
// platform, common/kdtree.c:569-570), by a bitonic sort of (distsq, index)
// keys in LDS; then obs_findlocal's selection (observations.c:1899-1908):
// the first min(n, NLOBSMAX) candidates, skipping those whose status is not
// OK.  Writes the sorted candidates and the list length.  Lists of more
// than kSortMax candidates are loc_sort_big_kernel's.
constexpr int kSortMax = 8192;

__global__ void __launch_bounds__(256) loc_sort_kernel(int nnode, const TypeInfo* __restrict__ types, int ntypes,
                                                       const short* __restrict__ status,
                                                       const int* __restrict__ raw,
                                                       const long long* __restrict__ rawoff,
                                                       const int* __restrict__ rrow, const double* __restrict__ rd2,
                                                       int* __restrict__ srow, double* __restrict__ sd2,
                                                       int* __restrict__ counts)
{
    __shared__ double kd[kSortMax];
    __shared__ int ki[kSortMax];
    __shared__ int cnt;
    const long long item = blockIdx.x;
    if (item >= (long long)nnode * ntypes)
        return;
    const int n = raw[item];
    if (n == 0 || n > kSortMax)
        return;
    const TypeInfo& ti = types[item % ntypes];
    const long long off = rawoff[item];
    int P = 1;
    while (P < n)
        P <<= 1;
    for (int k = threadIdx.x; k < P; k += 256) {
        kd[k] = (k < n) ? rd2[off + k] : INFINITY;
        ki[k] = k;
    }
    if (threadIdx.x == 0)
        cnt = 0;
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int k = threadIdx.x; k < P / 2; k += 256) {
                const int lo = 2 * stride * (k / stride) + (k % stride);
                const int hi = lo + stride;
                const bool up = ((lo & size) == 0);
                const double a = kd[lo], b = kd[hi];
                const int ia = ki[lo], ib = ki[hi];
                const bool agt = (a > b) || (a == b && ia > ib);
                if (agt == up) {
                    kd[lo] = b;
                    kd[hi] = a;
                    ki[lo] = ib;
                    ki[hi] = ia;
                }
            }
            __syncthreads();
        }
    }
    const int nsel = min(n, ti.nlobsmax);
    int mine = 0;
    for (int k = threadIdx.x; k < n; k += 256) {
        const int row = rrow[off + ki[k]];
        srow[off + k] = row;
        sd2[off + k] = kd[k];
        if (k < nsel && status[row] == kStatusOK)
            mine++;
    }
    atomicAdd(&cnt, mine);
    __syncthreads();
    if (threadIdx.x == 0)
        counts[item] = cnt;
}

// Lists of more than kSortMax candidates (the reference has no limit): one
// workgroup sorts a (node, type)'s candidates in place in global memory by a
// bottom-up merge sort on the squared distance, stable -- equal distances
// keep their visiting order, the order loc_sort_kernel's (distance, index)
// keys give -- ping-ponging between (rd2, rrow) and (sd2, srow); each
// element finds its place in the merged run by a binary search in the other
// run.  Then the same selection.
__global__ void __launch_bounds__(256) loc_sort_big_kernel(int nnode, const TypeInfo* __restrict__ types,
                                                           int ntypes, const short* __restrict__ status,
                                                           const int* __restrict__ raw,
                                                           const long long* __restrict__ rawoff, int* __restrict__ rrow,
                                                           double* __restrict__ rd2, int* __restrict__ srow,
                                                           double* __restrict__ sd2, int* __restrict__ counts)
{
    __shared__ int cnt;
    const long long item = blockIdx.x;
    if (item >= (long long)nnode * ntypes)
        return;
    const int n = raw[item];
    if (n <= kSortMax)
        return;
    const TypeInfo& ti = types[item % ntypes];
    const long long off = rawoff[item];
    double* keys[2] = {rd2 + off, sd2 + off};
    int* rows[2] = {rrow + off, srow + off};
    int src = 0;
    for (int width = 1; width < n; width <<= 1) {
        const double* ik = keys[src];
        const int* ir = rows[src];
        double* ok = keys[src ^ 1];
        int* orow = rows[src ^ 1];
        for (int k = threadIdx.x; k < n; k += 256) {
            const int r0 = (k / (2 * width)) * (2 * width);   // the pair of runs [r0, mid) [mid, end)
            const int mid = min(r0 + width, n), end = min(r0 + 2 * width, n);
            const double key = ik[k];
            int pos;
            if (k < mid) {   // before the right run's elements >= key
                int lo = mid, hi = end;
                while (lo < hi) {
                    const int h = (lo + hi) >> 1;
                    if (ik[h] < key)
                        lo = h + 1;
                    else
                        hi = h;
                }
                pos = k + (lo - mid);
            } else {         // after the left run's elements <= key
                int lo = r0, hi = mid;
                while (lo < hi) {
                    const int h = (lo + hi) >> 1;
                    if (ik[h] <= key)
                        lo = h + 1;
                    else
                        hi = h;
                }
                pos = (k - mid) + lo;
            }
            ok[pos] = key;
            orow[pos] = ir[k];
        }
        __syncthreads();   // the pass is complete before the next reads it
        src ^= 1;
    }
    if (src == 0) {   // the sorted candidates end in (sd2, srow)
        for (int k = threadIdx.x; k < n; k += 256) {
            sd2[off + k] = rd2[off + k];
            srow[off + k] = rrow[off + k];
        }
    }
    if (threadIdx.x == 0)
        cnt = 0;
    __syncthreads();
    const int nsel = min(n, ti.nlobsmax);
    int mine = 0;
    for (int k = threadIdx.x; k < nsel; k += 256)
        if (status[srow[off + k]] == kStatusOK)
            mine++;
    atomicAdd(&cnt, mine);
    __syncthreads();
    if (threadIdx.x == 0)
        counts[item] = cnt;
}

// Fills the lists in the reference's order (walked in the tree).  Each thread
// keeps its entries in registers and writes them as runs that end on a
// multiple of kLocBurst (32 bytes of ids, 64 of tapers): single 4- and 8-byte
// stores from 64 threads walking different lists leave their cache lines
// part-written, and such lines are written back to memory several times over
// (174 against 105 ms per localisation of the 51x1500x1800 tile; runs of 4
// gave 118 ms, of 16 106 ms).  nnode nodes from node0; ids and lc start at list
// entry off0 (a multiple of kLocBurst).
//
// Few lists (lanes > 0): `lanes` of them in a row per wavefront instead of a
// tile, so that they spread over kFillWaves wavefronts.  A wavefront's step
// waits for the slowest of its lanes' loads, and a few wavefronts hide none of
// it: 9 nodes of four types 13 -> 5.7 ms (512 to 8,192 wavefronts alike), 1,024
// nodes 16.7 -> 8.9 ms (512: 10.7, 8,192: 7.4).
constexpr int kLocBurst = 8;
constexpr int kFillWaves = 2048;
constexpr int kFillLanes = 8;   // beyond that, tiles

__global__ void __launch_bounds__(64) loc_fill_kernel(int nnode, int ni, const double* __restrict__ qxyz,
                                                       const unsigned char* __restrict__ isglobal,
                                                       const unsigned char* __restrict__ visible,
                                                       const KdNode* __restrict__ nodes,
                                                       const int* __restrict__ noderow,
                                                       const TypeInfo* __restrict__ types, int ntypes,
                                                       const short* __restrict__ status,
                                                       const int* __restrict__ obsids,
                                                       const long long* __restrict__ offsets, int* __restrict__ ids,
                                                       double* __restrict__ lc, const long long* __restrict__ rawoff,
                                                       const int* __restrict__ raw, const int* __restrict__ srow,
                                                       const double* __restrict__ sd2, int node0, long long off0, int lanes)
{
    int t, node;
    if (lanes == 0) {
        if (!thread_node(nnode, ni, ntypes, t, node))
            return;
    } else {
        const long long it = (long long)blockIdx.x * lanes + threadIdx.x;
        if ((int)threadIdx.x >= lanes || it >= (long long)nnode * ntypes)
            return;
        t = (int)(it / nnode);
        node = (int)(it - (long long)t * nnode);
    }
    node += node0;
    double q[3] = {qxyz[3 * (size_t)node], qxyz[3 * (size_t)node + 1], qxyz[3 * (size_t)node + 2]};
    const bool glob = isglobal[node] != 0;
    const TypeInfo& ti = types[t];
    if (!ti.searchable || !(visible == nullptr || visible[t]))
        return;
    long long o = offsets[(size_t)node * ntypes + t] - off0;
    if (glob) {
        for (int i = 0; i < ti.nids; ++i) {
            ids[o + i] = obsids[ti.obsid0 + i];
            lc[o + i] = 1.0;
        }
    } else if (ti.nnode > 0 && ti.nlobsmax != ENKFG_NLOBSMAX_NONE) {
        const size_t item = (size_t)node * ntypes + t;
        const long long r0 = rawoff[item];
        const int nsel = min(raw[item], ti.nlobsmax);
        for (int k = 0; k < nsel; ++k) {
            const int row = srow[r0 + k];
            if (status[row] == kStatusOK) {
                ids[o] = row;
                lc[o] = calclcoeff(ti, sqrt(sd2[r0 + k]));
                o++;
            }
        }
    } else if (ti.nnode > 0) {
        int bid[kLocBurst];
        double blc[kLocBurst];
#pragma unroll
        for (int b = 0; b < kLocBurst; ++b) {
            bid[b] = 0;
            blc[b] = 0.0;
        }
        long long first = o;   // entries first .. o - 1 are in the registers, entry e at e % kLocBurst
        range_walk(nodes + ti.node0, ti.ndim, q, ti.range, [&](int v, double distsq) {
            const int row = noderow[ti.node0 + v];   // device row of the node's observation
            if (status[row] != kStatusOK)
                return;
            const double c = calclcoeff(ti, sqrt(distsq));
            const int nb = (int)(o % kLocBurst);
#pragma unroll
            for (int b = 0; b < kLocBurst; ++b) {
                bid[b] = (b == nb) ? row : bid[b];
                blc[b] = (b == nb) ? c : blc[b];
            }
            ++o;
            if (nb == kLocBurst - 1) {
                const long long w = o - kLocBurst;   // a multiple of kLocBurst
                if (first <= w) {
                    int4* di = reinterpret_cast<int4*>(ids + w);
                    double2* dl = reinterpret_cast<double2*>(lc + w);
#pragma unroll
                    for (int b = 0; b < kLocBurst; b += 4)
                        di[b / 4] = make_int4(bid[b], bid[b + 1], bid[b + 2], bid[b + 3]);
#pragma unroll
                    for (int b = 0; b < kLocBurst; b += 2)
                        dl[b / 2] = make_double2(blc[b], blc[b + 1]);
                } else {   // the list starts inside this run
#pragma unroll
                    for (int b = 0; b < kLocBurst; ++b)
                        if (w + b >= first) {
                            ids[w + b] = bid[b];
                            lc[w + b] = blc[b];
                        }
                }
                first = o;
            }
        });
        const long long w = o - o % kLocBurst;
#pragma unroll
        for (int b = 0; b < kLocBurst; ++b)
            if (w + b >= first && w + b < o) {
                ids[w + b] = bid[b];
                lc[w + b] = blc[b];
            }
    }
}

// ---------------------------------------------------------------- box search
//
// One wavefront per (node, obstype).  FILL == false counts the lists; FILL ==
// true, given the scanned offsets, writes them: hits are gathered in LDS and
// written 64 at a time, so that the tapers are computed with every lane busy
// and the stores are whole runs.  kBoxAhead leaves are loaded together, since
// a step's loads, from L2 or beyond, are its latency.
constexpr int kBoxAhead = 4;
// consecutive blocks (of four items) per XCD run: four 8 x 8 tiles of nodes
constexpr int kBoxRun = 64;

// Item `it` as (type, node): 64 consecutive items are an 8 x 8 tile of the
// stride grid and one type, so the wavefronts in flight on an XCD search a
// compact patch.  ok is false past the grid's edge.
__device__ inline bool box_item(long long it, int ni, int nj, int ntypes, int& t, int& node)
{
    const int ti = (ni + 7) / 8, tj = (nj + 7) / 8;
    const long long per_type = (long long)ti * tj * 64;
    if (it >= per_type * ntypes)
        return false;
    t = (int)(it / per_type);
    const long long rem = it - (long long)t * per_type;
    const int tile = (int)(rem / 64), k = (int)(rem % 64);
    const int i = (tile % ti) * 8 + k % 8, j = (tile / ti) * 8 + k / 8;
    if (i >= ni || j >= nj)
        return false;
    node = j * ni + i;
    return true;
}

template <int ND>
__device__ inline double box_distsq(const LocBox& b, double q0, double q1, double q2)
{
    // the distance of the nearest point of the box, summed as distsq is; the
    // difference to a face, and 0 inside
    double s = 0.0;
    double d = fmax(fmax((double)b.lo[0] - q0, q0 - (double)b.hi[0]), 0.0);
    s += d * d;
    d = fmax(fmax((double)b.lo[1] - q1, q1 - (double)b.hi[1]), 0.0);
    s += d * d;
    if (ND == 3) {
        d = fmax(fmax((double)b.lo[2] - q2, q2 - (double)b.hi[2]), 0.0);
        s += d * d;
    }
    return s;
}

// orders the LDS accesses of one wavefront
__device__ inline void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Does the tree walk reach node v?  Every ancestor must have led to v's side:
// its near one, or the far one if the range crosses the split (range_walk_nd).
template <int ND>
__device__ inline bool walk_reaches(const KdNode* __restrict__ tree, int v, double range, double q0, double q1, double q2)
{
    int depth = 0;
    for (int p = (int)(tree[v].link & 0x7fffffffu) - 1; p >= 0; p = (int)(tree[p].link & 0x7fffffffu) - 1)
        ++depth;
    while (depth > 0) {
        const int p = (int)(tree[v].link & 0x7fffffffu) - 1;
        const KdNode nd = tree[p];
        const int dir = --depth % ND;
        const double cd = dir == 0 ? nd.x : ((ND == 2 || dir == 1) ? nd.y : nd.z);
        const double qd = dir == 0 ? q0 : ((ND == 2 || dir == 1) ? q1 : q2);
        const double dx = qd - cd;
        const bool left = (nd.link & 0x80000000u) && v == p + 1;
        if (left != (dx <= 0.0) && !(fabs(dx) < range))
            return false;
        v = p;
    }
    return true;
}

// TREES: observations a whole range away along an axis climb their tree; else
// counting sets tie for them (and there are none when the lists are filled)
template <int ND, bool FILL, bool TREES>
__device__ inline int box_search(const TypeInfo& ti, const LocBox* __restrict__ boxes, const double* __restrict__ xyz,
                                 size_t nrow, const short* __restrict__ status, const KdNode* __restrict__ nodes,
                                 const int* __restrict__ rownode, const double* q, int* __restrict__ ids,
                                 double* __restrict__ lc, double* sd, int* si, bool& tie)
{
    const int lane = threadIdx.x & 63;
    const double q0 = q[0], q1 = q[1], q2 = ND == 3 ? q[2] : 0.0;
    const double r2 = ti.range * ti.range;
    const LocBox* __restrict__ L1 = boxes + ti.box0[0];
    const LocBox* __restrict__ L2 = boxes + ti.box0[1];
    const LocBox* __restrict__ L3 = boxes + ti.box0[2];
    const double* __restrict__ X = xyz;
    const double* __restrict__ Y = xyz + nrow;
    const double* __restrict__ Z = xyz + 2 * nrow;
    const unsigned long long below = (1ULL << lane) - 1ULL;
    const int row0 = ti.node0, row1 = ti.node0 + ti.nnode;
    int n = 0;       // entries counted, or written
    int nbuf = 0;    // entries in LDS
    for (int c3 = 0; c3 < ti.nbox[2]; c3 += 64) {
        const int b3 = c3 + lane;
        unsigned long long h3 =
            __ballot(b3 < ti.nbox[2] && !(box_distsq<ND>(L3[min(b3, ti.nbox[2] - 1)], q0, q1, q2) > r2));
        while (h3) {
            const int p3 = c3 + __builtin_ctzll(h3);
            h3 &= h3 - 1;
            const int b2 = p3 * 64 + lane;
            unsigned long long h2 =
                __ballot(b2 < ti.nbox[1] && !(box_distsq<ND>(L2[min(b2, ti.nbox[1] - 1)], q0, q1, q2) > r2));
            while (h2) {
                const int p2 = p3 * 64 + __builtin_ctzll(h2);
                h2 &= h2 - 1;
                const int b1 = p2 * 64 + lane;
                unsigned long long h1 =
                    __ballot(b1 < ti.nbox[0] && !(box_distsq<ND>(L1[min(b1, ti.nbox[0] - 1)], q0, q1, q2) > r2));
                while (h1) {
                    int row[kBoxAhead];
                    double x[kBoxAhead], y[kBoxAhead], z[kBoxAhead];
                    short st[kBoxAhead];
#pragma unroll
                    for (int u = 0; u < kBoxAhead; ++u) {
                        // past the last hit leaf: a row beyond the type's
                        row[u] = h1 ? row0 + (p2 * 64 + __builtin_ctzll(h1)) * 64 + lane : row1;
                        h1 = h1 ? (h1 & (h1 - 1)) : 0ULL;
                        const int r = min(row[u], row1 - 1);
                        x[u] = X[r];
                        y[u] = Y[r];
                        z[u] = ND == 3 ? Z[r] : 0.0;
                        st[u] = status[r];
                    }
                    double dsq[kBoxAhead];
                    bool ok[kBoxAhead], at = false;
                    const auto test = [&](int u) {
                        // kd_findnodeswithinrange's sum, in its order (kdtree.c:529-533)
                        double distsq = 0.0;
                        double d = x[u] - q0;
                        distsq += d * d;
                        d = y[u] - q1;
                        distsq += d * d;
                        if (ND == 3) {
                            d = z[u] - q2;
                            distsq += d * d;
                        }
                        dsq[u] = distsq;
                        ok[u] = row[u] < row1 && distsq <= r2 && st[u] == kStatusOK;
                        at |= ok[u] && distsq == r2;
                    };
                    const auto put = [&](int u) {
                        const unsigned long long m = __ballot(ok[u]);
                        if (!FILL) {
                            n += __popcll(m);
                        } else if (m) {
                            if (ok[u]) {
                                const int pos = nbuf + __popcll(m & below);
                                sd[pos] = dsq[u];
                                si[pos] = row[u];
                            }
                            nbuf += __popcll(m);
                            wave_lds_fence();
                            if (nbuf >= 64) {
                                ids[n + lane] = si[lane];
                                lc[n + lane] = calclcoeff(ti, sqrt(sd[lane]));
                                n += 64;
                                nbuf -= 64;
                                const double td = sd[64 + lane];
                                const int tr = si[64 + lane];
                                wave_lds_fence();
                                sd[lane] = td;
                                si[lane] = tr;
                                wave_lds_fence();
                            }
                        }
                    };
                    if (FILL && !TREES) {
#pragma unroll
                        for (int u = 0; u < kBoxAhead; ++u) {
                            test(u);
                            put(u);
                        }
                        continue;
                    }
#pragma unroll
                    for (int u = 0; u < kBoxAhead; ++u)
                        test(u);
                    if (__builtin_expect(__ballot(at) != 0, 0)) {
                        // at exactly the range: where all of it is along one
                        // axis the walk may have pruned it
                        unsigned ties = 0, pruned = 0;
#pragma unroll
                        for (int u = 0; u < kBoxAhead; ++u)
                            ties |= (ok[u] && dsq[u] == r2) ? 1u << u : 0u;
#pragma unroll 1
                        for (int v = 0; v < kBoxAhead; ++v) {
                            if (!((ties >> v) & 1))
                                continue;
                            int r = row0;
#pragma unroll
                            for (int u = 0; u < kBoxAhead; ++u)
                                r = u == v ? row[u] : r;
                            if (!(fabs(X[r] - q0) >= ti.range || fabs(Y[r] - q1) >= ti.range ||
                                  (ND == 3 && fabs(Z[r] - q2) >= ti.range)))
                                continue;
                            if (!TREES)
                                tie = true;
                            else if (!walk_reaches<ND>(nodes + ti.node0, rownode[r], ti.range, q0, q1, q2))
                                pruned |= 1u << v;
                        }
#pragma unroll
                        for (int u = 0; u < kBoxAhead; ++u)
                            ok[u] = ok[u] && !((pruned >> u) & 1);
                    }
#pragma unroll
                    for (int u = 0; u < kBoxAhead; ++u)
                        put(u);
                }
            }
        }
    }
    if (FILL && lane < nbuf) {
        ids[n + lane] = si[lane];
        lc[n + lane] = calclcoeff(ti, sqrt(sd[lane]));
    }
    return n;
}

template <bool FILL, bool TREES>
__global__ void __launch_bounds__(256) loc_box_kernel(int ni, int nj, const double* __restrict__ qxyz,
                                                      const unsigned char* __restrict__ isglobal,
                                                      const unsigned char* __restrict__ visible,
                                                      const TypeInfo* __restrict__ types, int ntypes,
                                                      const LocBox* __restrict__ boxes,
                                                      const double* __restrict__ xyz, size_t nrow,
                                                      const short* __restrict__ status, const int* __restrict__ obsids,
                                                      const KdNode* __restrict__ nodes, const int* __restrict__ rownode,
                                                      int* __restrict__ counts, const long long* __restrict__ offsets,
                                                      int* __restrict__ ids, double* __restrict__ lc,
                                                      int* __restrict__ tieflag, unsigned run0)
{
    __shared__ double sd[FILL ? 4 * 128 : 1];
    __shared__ int si[FILL ? 4 * 128 : 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned s = blockIdx.x / 8, x = blockIdx.x % 8;
    const long long blk = ((long long)(run0 + s / kBoxRun) * 8 + x) * kBoxRun + s % kBoxRun;
    int t, node;
    if (!box_item(blk * 4 + wave, ni, nj, ntypes, t, node))
        return;
    t = __builtin_amdgcn_readfirstlane(t);   // one item per wavefront
    node = __builtin_amdgcn_readfirstlane(node);
    const TypeInfo& ti = types[t];
    const size_t item = (size_t)node * ntypes + t;
    int n = 0;
    if (ti.searchable && (visible == nullptr || visible[t])) {
        const long long o = FILL ? offsets[item] : 0;
        if (isglobal[node]) {
            n = ti.nids;   // obs_getglobal: all obs of the type, no status check
            if (FILL)
                for (int i = lane; i < n; i += 64) {
                    ids[o + i] = obsids[ti.obsid0 + i];
                    lc[o + i] = 1.0;
                }
        } else if (ti.nnode > 0) {
            const double q[3] = {qxyz[3 * (size_t)node], qxyz[3 * (size_t)node + 1], qxyz[3 * (size_t)node + 2]};
            bool tie = false;
            double* wsd = FILL ? sd + wave * 128 : nullptr;
            int* wsi = FILL ? si + wave * 128 : nullptr;
            int* wid = FILL ? ids + o : nullptr;
            double* wlc = FILL ? lc + o : nullptr;
            n = ti.ndim == 3
                    ? box_search<3, FILL, TREES>(ti, boxes, xyz, nrow, status, nodes, rownode, q, wid, wlc, wsd, wsi, tie)
                    : box_search<2, FILL, TREES>(ti, boxes, xyz, nrow, status, nodes, rownode, q, wid, wlc, wsd, wsi, tie);
            if (!FILL && !TREES && __ballot(tie) && lane == 0)
                atomicExch(tieflag, 1);
        }
    }
    if (!FILL && lane == 0)
        counts[item] = n;
}

// ---- exclusive scan of int counts into long long offsets (n + 1 entries)
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanChunk = kScanThreads * kScanItems;

__device__ inline long long block_exclusive_scan(long long v, long long* sh, long long* total)
{
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int off = 1; off < kScanThreads; off <<= 1) {
        long long add = (tid >= off) ? sh[tid - off] : 0;
        __syncthreads();
        sh[tid] += add;
        __syncthreads();
    }
    long long incl = sh[tid];
    *total = sh[kScanThreads - 1];
    __syncthreads();
    return incl - v;
}

__global__ void __launch_bounds__(kScanThreads) scan_partials_kernel(const int* __restrict__ in, long long n,
                                                                    long long* __restrict__ partials)
{
    __shared__ long long sh[kScanThreads];
    const long long base = (long long)blockIdx.x * kScanChunk;
    long long sum = 0;
    for (int k = 0; k < kScanItems; ++k) {
        long long i = base + (long long)threadIdx.x * kScanItems + k;
        if (i < n)
            sum += in[i];
    }
    long long total;
    block_exclusive_scan(sum, sh, &total);
    if (threadIdx.x == 0)
        partials[blockIdx.x] = total;
}

__global__ void __launch_bounds__(kScanThreads) scan_top_kernel(long long* __restrict__ partials, int nb)
{
    __shared__ long long sh[kScanThreads];
    long long carry = 0;
    for (int b0 = 0; b0 < nb; b0 += kScanThreads) {
        int i = b0 + threadIdx.x;
        long long v = (i < nb) ? partials[i] : 0;
        long long total;
        long long ex = block_exclusive_scan(v, sh, &total);
        if (i < nb)
            partials[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0)
        partials[nb] = carry;
}

__global__ void __launch_bounds__(kScanThreads) scan_final_kernel(const int* __restrict__ in, long long n,
                                                                 const long long* __restrict__ partials,
                                                                 long long* __restrict__ out, int nb)
{
    __shared__ long long sh[kScanThreads];
    const long long base = (long long)blockIdx.x * kScanChunk;
    long long vals[kScanItems];
    long long sum = 0;
    for (int k = 0; k < kScanItems; ++k) {
        long long i = base + (long long)threadIdx.x * kScanItems + k;
        vals[k] = (i < n) ? in[i] : 0;
        sum += vals[k];
    }
    long long total;
    long long ex = block_exclusive_scan(sum, sh, &total) + partials[blockIdx.x];
    for (int k = 0; k < kScanItems; ++k) {
        long long i = base + (long long)threadIdx.x * kScanItems + k;
        if (i < n)
            out[i] = ex;
        ex += vals[k];
    }
    if (blockIdx.x == nb - 1 && threadIdx.x == 0)
        out[n] = partials[nb];
}

// grid of the walk kernels: one 64-thread block per 8 x 8 tile and obstype
// (thread_node), rounded up to a multiple of 8 runs
inline dim3 walk_grid(int ni, int nj, int ntypes)
{
    const long long n = (long long)ntypes * (((ni + 7) / 8 + 7) / 8) * (((nj + 7) / 8 + 7) / 8) * 64;
    return dim3((unsigned)(8 * kWalkRun * ((n + 8 * kWalkRun - 1) / (8 * kWalkRun))));
}

}  // namespace

hipError_t launch_loc_count(hipStream_t s, int ni, int nj, const double* qxyz, const unsigned char* isglobal,
                            const unsigned char* visible, const KdNode* nodes, const int* noderow,
                            const TypeInfo* types, int ntypes,
                            const short* status, int* counts, int* raw)
{
    const long long nt = (long long)ni * nj * ntypes;
    if (nt <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(loc_count_kernel, walk_grid(ni, nj, ntypes), dim3(64), 0, s, ni * nj, ni, qxyz, isglobal,
                       visible, nodes, noderow, types, ntypes, status, counts, raw);
    return hipGetLastError();
}

hipError_t launch_loc_nlobsmax(hipStream_t s, int ni, int nj, const double* qxyz, const unsigned char* isglobal,
                               const unsigned char* visible, const KdNode* nodes, const int* noderow,
                            const TypeInfo* types, int ntypes,
                               const short* status, const int* raw, const long long* rawoff, int* rrow, double* rd2,
                               int* srow, double* sd2, int* counts)
{
    const long long nt = (long long)ni * nj * ntypes;
    if (nt <= 0)
        return hipSuccess;
    if (nt > 0x7fffffffLL)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(loc_rawfill_kernel, walk_grid(ni, nj, ntypes), dim3(64), 0, s, ni * nj, ni, qxyz, isglobal,
                       visible, nodes, noderow, types, ntypes, rawoff, rrow, rd2);
    hipLaunchKernelGGL(loc_sort_kernel, dim3((unsigned)nt), dim3(256), 0, s, ni * nj, types, ntypes, status, raw,
                       rawoff, rrow, rd2, srow, sd2, counts);
    hipLaunchKernelGGL(loc_sort_big_kernel, dim3((unsigned)nt), dim3(256), 0, s, ni * nj, types, ntypes, status, raw,
                       rawoff, rrow, rd2, srow, sd2, counts);
    return hipGetLastError();
}

hipError_t launch_loc_fill(hipStream_t s, int ni, int nj, const double* qxyz, const unsigned char* isglobal,
                           const unsigned char* visible, const KdNode* nodes, const int* noderow,
                           const TypeInfo* types, int ntypes, const short* status, const int* obsids,
                           const long long* offsets, int* ids, double* lc, const long long* rawoff, const int* raw,
                           const int* srow, const double* sd2, int node0, int n, long long off0)
{
    const bool all = n == 0;
    const long long nn = all ? (long long)ni * nj : n, nt = nn * ntypes;
    if (nt <= 0)
        return hipSuccess;
    if (off0 % kLocBurst != 0)
        return hipErrorInvalidValue;
    const int lanes = (int)std::min<long long>((nt + kFillWaves - 1) / kFillWaves, 64);
    if (all && lanes > kFillLanes)
        hipLaunchKernelGGL(loc_fill_kernel, walk_grid(ni, nj, ntypes), dim3(64), 0, s, ni * nj, ni, qxyz, isglobal,
                           visible, nodes, noderow, types, ntypes, status, obsids, offsets, ids, lc, rawoff, raw, srow,
                           sd2, 0, 0LL, 0);
    else
        hipLaunchKernelGGL(loc_fill_kernel, dim3((unsigned)((nt + lanes - 1) / lanes)), dim3(64), 0, s, (int)nn, ni,
                           qxyz, isglobal, visible, nodes, noderow, types, ntypes, status, obsids, offsets, ids, lc,
                           rawoff, raw, srow, sd2, node0, off0, lanes);
    return hipGetLastError();
}

// tmp must hold (nb + 1) long longs, nb = ceil(n / 2048); with tmp == nullptr
// the required size is returned in *tmp_bytes.
hipError_t launch_scan_counts(hipStream_t s, const int* counts, long long* offsets, long long n, void* tmp,
                              size_t* tmp_bytes)
{
    const long long nb = (n + kScanChunk - 1) / kScanChunk;
    const size_t need = (size_t)(nb + 1) * sizeof(long long);
    if (tmp == nullptr) {
        *tmp_bytes = need;
        return hipSuccess;
    }
    if (*tmp_bytes < need)
        return hipErrorInvalidValue;
    long long* partials = static_cast<long long*>(tmp);
    if (n == 0) {
        // offsets[0] = 0 via the top kernel with nb = 0
        hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(kScanThreads), 0, s, offsets, 0);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(scan_partials_kernel, dim3((unsigned)nb), dim3(kScanThreads), 0, s, counts, n, partials);
    hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(kScanThreads), 0, s, partials, (int)nb);
    hipLaunchKernelGGL(scan_final_kernel, dim3((unsigned)nb), dim3(kScanThreads), 0, s, counts, n, partials, offsets,
                       (int)nb);
    return hipGetLastError();
}

hipError_t launch_loc_box(hipStream_t s, int ni, int nj, const double* qxyz, const unsigned char* isglobal,
                          const unsigned char* visible, const TypeInfo* types, int ntypes, const LocBox* boxes,
                          const double* xyz, size_t nrow, const short* status, const int* obsids,
                          const KdNode* nodes, const int* rownode, int* counts, int* tieflag,
                          const long long* offsets, int* ids, double* lc)
{
    if ((long long)ni * nj * ntypes <= 0)
        return hipSuccess;
    const long long blocks = (long long)((ni + 7) / 8) * ((nj + 7) / 8) * 16 * ntypes;
    const long long round = 8LL * kBoxRun;
    const long long rounds = (blocks + round - 1) / round;
    if (rounds > 0xffffffffLL)
        return hipErrorInvalidValue;
    // a launch holds fewer than 2^32 threads: 16M blocks, 64M lists
    constexpr long long per = (1LL << 24) / (8 * kBoxRun) - 1;
    for (long long r0 = 0; r0 < rounds; r0 += per) {
        const dim3 grid((unsigned)(round * std::min(per, rounds - r0)));
        const auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, ni, nj, qxyz, isglobal, visible, types, ntypes, boxes, xyz,
                               nrow, status, obsids, nodes, rownode, counts, offsets, ids, lc, tieflag, (unsigned)r0);
        };
        if (nodes == nullptr)
            ids == nullptr ? launch(loc_box_kernel<false, false>) : launch(loc_box_kernel<true, false>);
        else
            ids == nullptr ? launch(loc_box_kernel<false, true>) : launch(loc_box_kernel<true, true>);
    }
    return hipGetLastError();
}

}  // namespace enkfg
