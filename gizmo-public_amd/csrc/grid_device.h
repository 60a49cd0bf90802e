// grid_device.h -- device helpers shared by the stage kernels: launch
// geometry, the cell-grid walk, the periodic wrap and wavefront reductions.
#pragma once

#include <type_traits>

#include "gzm_internal.h"

namespace gzm {

// Call a walk's visitor; a visitor returning bool stops the walk with false.
template <typename F, typename... A>
__device__ __forceinline__ bool visit_more(F &f, A... args)
{
    if constexpr (std::is_void_v<decltype(f(args...))>) {
        f(args...);
        return true;
    } else {
        return f(args...);
    }
}

constexpr int kBlock = 256;
// largest workgroup of the per-particle loop kernels (density sweeps,
// gradients, the pair-list force loops), whose size gzm_params.block_size
// picks from 64, 128, 256 and 512 per stage.  The scanning force kernels stay
// at 256: a bound of 512 threads makes the compiler fit their 256 VGPRs to two
// waves per SIMD, with 3-5x the spills.
constexpr int kMaxBlock = 512;
constexpr int kXcds = 8;         // MI355X: 8 XCDs, each with its own L2
constexpr int kListChunk = 16;   // pair-list entries a lane stages before one 64-byte store
static_assert(kDensityCacheCap % kListChunk == 0, "a row's last chunk would reach into the next row");

// Workgroups are dealt to the XCDs round-robin (block b runs on XCD b % 8).
// Renumber them so that each XCD receives one contiguous run of the
// Morton-ordered particles: its L2 then holds the cells its waves share,
// instead of every eighth block of the whole box.  A bijection on
// [0, gridDim.x) for any grid size.
__device__ __forceinline__ int xcd_block()
{
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    const int q = nb / kXcds, r = nb % kXcds, x = b % kXcds;
    return x * q + (x < r ? x : r) + b / kXcds;
}

__device__ __forceinline__ int cell_coord(double x, double inv_s, int nc)
{
    int c = (int)floor(x * inv_s);
    if (c < 0) c = 0;
    if (c >= nc) c = nc - 1;
    return c;
}

__device__ __forceinline__ uint32_t spread10(uint32_t v)
{
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t morton3(int cx, int cy, int cz)
{
    return (spread10((uint32_t)cx) << 2) | (spread10((uint32_t)cy) << 1) | spread10((uint32_t)cz);
}

__device__ __forceinline__ double axis_gap(double x, double c0, double s)
{
    double g = c0 - x;
    double g2 = x - (c0 + s);
    g = (g > g2) ? g : g2;
    return (g > 0) ? g : 0.0;
}

// Visit every cell that may hold a particle within distance R of (x, y, z),
// periodic; cells whose box lies farther than R are skipped.  f(cx, cy, cz,
// begin, end) receives the cell's unwrapped coordinates (outside [0, nc) when
// the walk crosses the periodic boundary; the image of a particle of that cell
// lies at x + (c - c_wrapped) * s) and its sorted slot range.  `full` reports
// the axes walked whole because R spans half the box.  An f returning bool
// ends the walk by returning false.  With h_pair >= 0 (pair searches: R is
// the box's max hsml) a cell farther than h_pair is visited only when its own
// max hsml reaches x: no particle of it can pair with x otherwise.
template <typename F>
__device__ __forceinline__ void for_each_cell(const Grid &g, const double xs[3], double R, bool full[3], F &&f,
                                              double h_pair = -1.0)
{
    int lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        // a radius that spans the axis (or is not finite) walks the whole axis once
        full[a] = !(R * g.inv_s[a] < 0.5 * g.nc[a] - 2.0);
        if (!full[a]) {
            lo[a] = (int)floor((xs[a] - R) * g.inv_s[a] - 1e-6);
            hi[a] = (int)floor((xs[a] + R) * g.inv_s[a] + 1e-6);
        } else {
            lo[a] = 0;
            hi[a] = g.nc[a] - 1;
        }
    }
    const double R2 = R * R * (1.0 + 1e-9);
    const double hp2 = h_pair * h_pair * (1.0 + 1e-9);
    for (int cx = lo[0]; cx <= hi[0]; ++cx) {
        const int wx = (cx < 0) ? cx + g.nc[0] : ((cx >= g.nc[0]) ? cx - g.nc[0] : cx);
        const double gx = full[0] ? 0.0 : axis_gap(xs[0], cx * g.s[0], g.s[0]);
        const double gx2 = gx * gx;
        if (gx2 > R2) continue;
        for (int cy = lo[1]; cy <= hi[1]; ++cy) {
            const int wy = (cy < 0) ? cy + g.nc[1] : ((cy >= g.nc[1]) ? cy - g.nc[1] : cy);
            const double gy = full[1] ? 0.0 : axis_gap(xs[1], cy * g.s[1], g.s[1]);
            const double gxy2 = gx2 + gy * gy;
            if (gxy2 > R2) continue;
            const int rowbase = (wx * g.nc[1] + wy) * g.nc[2];
            for (int cz = lo[2]; cz <= hi[2]; ++cz) {
                const int wz = (cz < 0) ? cz + g.nc[2] : ((cz >= g.nc[2]) ? cz - g.nc[2] : cz);
                const double gz = full[2] ? 0.0 : axis_gap(xs[2], cz * g.s[2], g.s[2]);
                const double d2 = gxy2 + gz * gz;
                if (d2 > R2) continue;
                if (h_pair >= 0 && d2 > hp2) {
                    const double hm = g.hmax[rowbase + wz];
                    if (d2 > hm * hm * (1.0 + 1e-9)) continue;
                }
                const int2 r = g.range[rowbase + wz];
                if (!visit_more(f, cx, cy, cz, r.x, r.y)) return;
            }
        }
    }
}

// for_each_cell's cells in the same order, consecutive cells of a z column
// joined where their slot ranges adjoin (the Morton order stores cells 2k and
// 2k + 1 of a column side by side): f(full, cx, cy, cz, begin, end) with the
// unwrapped coordinates of the first cell of the run; runs do not cross the
// periodic boundary.  An f returning false ends the walk.
template <typename F>
__device__ __forceinline__ void for_each_run(const Grid &g, const double xs[3], double R, F &&f)
{
    int lo[3], hi[3];
    bool full[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        full[a] = !(R * g.inv_s[a] < 0.5 * g.nc[a] - 2.0);
        lo[a] = full[a] ? 0 : (int)floor((xs[a] - R) * g.inv_s[a] - 1e-6);
        hi[a] = full[a] ? g.nc[a] - 1 : (int)floor((xs[a] + R) * g.inv_s[a] + 1e-6);
    }
    const double R2 = R * R * (1.0 + 1e-9), inv_R2 = 1.0 / R2;
    for (int cx = lo[0]; cx <= hi[0]; ++cx) {
        const int wx = (cx < 0) ? cx + g.nc[0] : ((cx >= g.nc[0]) ? cx - g.nc[0] : cx);
        const double gx = full[0] ? 0.0 : axis_gap(xs[0], cx * g.s[0], g.s[0]);
        const double gx2 = gx * gx;
        if (gx2 > R2) continue;
        for (int cy = lo[1]; cy <= hi[1]; ++cy) {
            const int wy = (cy < 0) ? cy + g.nc[1] : ((cy >= g.nc[1]) ? cy - g.nc[1] : cy);
            const double gy = full[1] ? 0.0 : axis_gap(xs[1], cy * g.s[1], g.s[1]);
            const double gxy2 = gx2 + gy * gy;
            if (gxy2 > R2) continue;
            const int2 *column = g.range + (wx * g.nc[1] + wy) * g.nc[2];
            // the cells in reach of this column, from the width of the sphere there
            int z0 = lo[2], z1 = hi[2];
            if (!full[2]) {
                const double w = R * ((double)__builtin_amdgcn_sqrtf((float)((R2 - gxy2) * inv_R2)) * (1 + 1e-6));
                z0 = max(z0, (int)floor((xs[2] - w) * g.inv_s[2] - 1e-6));
                z1 = min(z1, (int)floor((xs[2] + w) * g.inv_s[2] + 1e-6));
            }
            auto slots = [&](int cz) {
                if (cz > z1) return make_int2(0, 0);
                return column[(cz < 0) ? cz + g.nc[2] : ((cz >= g.nc[2]) ? cz - g.nc[2] : cz)];
            };
            int beg = 0, end = 0, first = 0;
            int2 r = slots(z0);
            // one step past the last cell hands over the last run
            for (int cz = z0; cz <= z1 + 1; ++cz) {
                const int2 next = slots(cz + 1);
                const int2 c = r;
                r = next;
                if (cz <= z1) {
                    if (c.x == c.y) continue;
                    if (c.x == end && end > beg && cz != 0 && cz != g.nc[2]) {
                        end = c.y;
                        continue;
                    }
                }
                if (end > beg && !f(full, cx, cy, first, beg, end)) return;
                beg = c.x;
                end = c.y;
                first = cz;
            }
        }
    }
}

// the votes of a group of W lanes, from bit 0
template <int W>
__device__ __forceinline__ uint64_t group_ballot(bool v)
{
    const uint64_t bits = __ballot(v);
    if constexpr (W == 64) return bits;
    else return (bits >> ((threadIdx.x & 63) & ~(W - 1))) & ((1ull << W) - 1);
}

// The candidates of W lanes of one particle (`sub` = 0 .. W - 1), a z column of
// cells for each lane: test(j, whole, cx, cy, cz) decides, hit(k, j) takes the hits
// with their rank k in the order of for_each_cell.  Returns their number; -1: a
// column held more hits than a lane keeps, or more than `limit` candidates.
constexpr int kColumnHits = 32;
template <int W, typename T, typename F>
__device__ __forceinline__ int for_columns(const Grid &g, const double xs[3], double R, int sub, int limit,
                                           int *kept /* kColumnHits of this lane, 256 apart */, T &&test, F &&hit)
{
    int lo[3], n[3];
    bool full[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        full[a] = !(R * g.inv_s[a] < 0.5 * g.nc[a] - 2.0);
        lo[a] = full[a] ? 0 : (int)floor((xs[a] - R) * g.inv_s[a] - 1e-6);
        n[a] = (full[a] ? g.nc[a] - 1 : (int)floor((xs[a] + R) * g.inv_s[a] + 1e-6)) - lo[a] + 1;
    }
    const double R2 = R * R * (1.0 + 1e-9);
    const bool whole = full[0] || full[1] || full[2];
    const int columns = n[0] * n[1];
    int total = 0, seen = 0;
    for (int c0 = 0; c0 < columns; c0 += W) {
        const int c = c0 + sub;
        int hits = 0;
        if (c < columns) {
            const int cx = lo[0] + c / n[1], cy = lo[1] + c % n[1];
            const double gx = full[0] ? 0.0 : axis_gap(xs[0], cx * g.s[0], g.s[0]);
            const double gy = full[1] ? 0.0 : axis_gap(xs[1], cy * g.s[1], g.s[1]);
            const double gxy2 = gx * gx + gy * gy;
            const int wx = (cx < 0) ? cx + g.nc[0] : ((cx >= g.nc[0]) ? cx - g.nc[0] : cx);
            const int wy = (cy < 0) ? cy + g.nc[1] : ((cy >= g.nc[1]) ? cy - g.nc[1] : cy);
            const int2 *column = g.range + (wx * g.nc[1] + wy) * g.nc[2];
            auto slots = [&](int cz) {
                if (cz >= lo[2] + n[2]) return make_int2(0, 0);
                const double gz = full[2] ? 0.0 : axis_gap(xs[2], cz * g.s[2], g.s[2]);
                if (gxy2 > R2 || gxy2 + gz * gz > R2) return make_int2(0, 0);
                return column[(cz < 0) ? cz + g.nc[2] : ((cz >= g.nc[2]) ? cz - g.nc[2] : cz)];
            };
            int2 r = slots(lo[2]);
            for (int z = 0; z < n[2]; z++) {
                const int2 next = slots(lo[2] + z + 1);  // under way while this cell is tested
                seen += r.y - r.x;
                if (seen > limit) break;
                for (int j = r.x; j < r.y; j += 4) {
                    bool in[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) in[k] = test(min(j + k, r.y - 1), whole, cx, cy, lo[2] + z) && j + k < r.y;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        if (in[k]) {
                            if (hits < kColumnHits) kept[256 * hits] = j + k;
                            hits++;
                        }
                }
                r = next;
            }
        }
        if (group_ballot<W>(hits > kColumnHits || seen > limit)) return -1;
        int sum = hits;
#pragma unroll
        for (int off = 1; off < W; off <<= 1) {
            const int o = __shfl_up(sum, off, W);
            if (sub >= off) sum += o;
        }
        for (int k = 0; k < hits; k++) hit(total + sum - hits + k, kept[256 * k]);
        total += __shfl(sum, W - 1, W);
    }
    return total;
}

// Visit every sorted slot k whose cell may hold a particle within distance R
// of (x, y, z), periodic.
template <typename F>
__device__ __forceinline__ void for_each_candidate(const Grid &g, const double xs[3], double R, F &&f,
                                                   double h_pair = -1.0)
{
    bool full[3];
    for_each_cell(g, xs, R, full, [&](int, int, int, int begin, int end) {
        for (int k = begin; k < end; ++k)
            if (!visit_more(f, k)) return false;
        return true;
    }, h_pair);
}

__device__ __forceinline__ void wrap_dp(const BoxInfo &box, double dp[3])
{
    dp[1] = wrap_axis(dp[1], box.L[1], box.half[1]);
    dp[0] = wrap_axis(dp[0], box.L[0], box.half[0]);
    dp[2] = wrap_axis(dp[2], box.L[2], box.half[2]);
}

// The same image for displacements whose nearest image is shorter than 0.45 of
// each side (BoxInfo::narrow2), in three instructions an axis instead of about
// ten: the multiple of L subtracted is 0 or +-L exactly, so dp rounds as in
// wrap_dp.  (A displacement near half a side may take the other image; it is
// longer than the caller's radius either way.)
__device__ __forceinline__ void wrap_near(const BoxInfo &box, double dp[3])
{
#pragma unroll
    for (int k = 0; k < 3; k++) dp[k] = fma(-rint(dp[k] * box.inv[k]), box.L[k], dp[k]);
}

// periodic distance from x to the interval [lo, hi] (both inside [0, L))
__device__ __forceinline__ double periodic_gap(double x, double lo, double hi, double L)
{
    double g = lo - x;
    const double g2 = x - hi;
    g = (g > g2) ? g : g2;
    g = (g > 0) ? g : 0.0;
    const double a = x + L - hi, b = lo + L - x;  // the images x + L, x - L
    g = (a < g) ? a : g;
    g = (b < g) ? b : g;
    return g;
}

// Visit (f(slot)) every particle of box G whose position may lie within R of
// x -- and, for the pair search, within the hsml of a particle below the
// node -- in depth-first Morton order.  Conservative by the same 1e-9
// relative margin as the cell walk; the caller applies the exact predicate.
// An f returning bool ends the walk by returning false.  One step per node or
// leaf (the walk the pair searches of the gradient and force loops use: their
// tree path is the rare one there, and the form below costs them registers).
template <typename F>
__device__ __forceinline__ void tree_walk(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                          bool pairs, F &&f)
{
    int node = G.root;
    // a well-formed tree visits each of its 2 count - 1 nodes at most once
    for (int steps = 2 * G.count; node != kTreeEnd && steps > 0; steps--) {
        if (node < 0) {
            const int j = -node - 1;
            if (!visit_more(f, j)) return;
            node = T.leaf_esc[j];
            continue;
        }
        const TreeNode nd = T.nodes[node];
        const double hm = nd.lo.w;
        const double Rn = (pairs && hm > R) ? hm : R;
        const double gx = periodic_gap(x[0], nd.lo.x, nd.hi.x, G.box.L[0]);
        const double gy = periodic_gap(x[1], nd.lo.y, nd.hi.y, G.box.L[1]);
        const double gz = periodic_gap(x[2], nd.lo.z, nd.hi.z, G.box.L[2]);
        const int esc = __float_as_int(nd.hi.w);
        if (!(gx * gx + gy * gy + gz * gz <= Rn * Rn * (1.0 + 1e-9))) {
            node = esc;
            continue;
        }
        if (nd.link.z - nd.link.y < kTreeBucket) {
            for (int j = nd.link.y; j <= nd.link.z; j++)
                if (!visit_more(f, j)) return;
            node = esc;
        } else {
            node = nd.link.x;
        }
    }
}

// The same visits as tree_walk (radius R only: the density search), in two
// nested loops ("while-while"): each lane walks nodes until it reaches a slot
// range to scan (a bucket or a single leaf), and the lanes then scan their
// ranges together.  In tree_walk's single loop a wavefront's lanes stand at
// nodes and buckets in no common rhythm, so nearly every step pays for a
// bucket scan (the candidate loop with its pair body) with the few lanes that
// happen to be at a bucket; here every unfinished lane is in the scan.  Each
// lane visits its candidates in the same order either way.
template <typename F>
__device__ __forceinline__ void tree_walk_grouped(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                                  F &&f)
{
    int node = G.root;
    int steps = 2 * G.count;  // as in tree_walk
    for (;;) {
        int beg = 0, end = -1;
        while (node != kTreeEnd && steps > 0) {
            steps--;
            if (node < 0) {
                beg = end = -node - 1;
                node = T.leaf_esc[beg];
                break;
            }
            const TreeNode nd = T.nodes[node];
            const double gx = periodic_gap(x[0], nd.lo.x, nd.hi.x, G.box.L[0]);
            const double gy = periodic_gap(x[1], nd.lo.y, nd.hi.y, G.box.L[1]);
            const double gz = periodic_gap(x[2], nd.lo.z, nd.hi.z, G.box.L[2]);
            const int esc = __float_as_int(nd.hi.w);
            if (!(gx * gx + gy * gy + gz * gz <= R * R * (1.0 + 1e-9))) {
                node = esc;
                continue;
            }
            if (nd.link.z - nd.link.y < kTreeBucket) {
                beg = nd.link.y;
                end = nd.link.z;
                node = esc;
                break;
            }
            node = nd.link.x;
        }
        if (beg > end) return;
        for (int j = beg; j <= end; j++)
            if (!visit_more(f, j)) return;
    }
}

// Every sorted slot that may hold a neighbour of x: the cell grid within R
// (pair search: R = max(h_i, box hmax)), or the tree (R = h_i, node hmax).
template <typename F>
__device__ __forceinline__ void for_each_neighbour_candidate(const TreeArgs &T, const BoxDesc &G,
                                                             const double x[3], double h_i, bool pairs, F &&f)
{
    if (T.nodes) {
        tree_walk(T, G, x, h_i, pairs, f);
    } else {
        const double R = (pairs && G.hmax > h_i) ? G.hmax : h_i;
        for_each_candidate(G.grid, x, R, f, pairs ? h_i : -1.0);
    }
}

// order this wavefront's LDS writes before its later reads
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// f(slot, valid) or f(slot, valid, last)
template <typename F>
__device__ __forceinline__ void walk_call(F &&f, int slot, bool valid, bool last)
{
    if constexpr (std::is_invocable<F, int, bool, bool>::value) f(slot, valid, last);
    else f(slot, valid);
}

// LDS of the tree walk of W lanes (group_tree_walk).  Past kWide entries fewer
// are taken at a time, in the end one by one, which adds at most an entry per
// level, and the 95 bits of a Morton key and slot bound the levels.  (Taking W
// from the end of the list adds up to W per level; at 5 W a dense clump's walk ran
// entry by entry.)
constexpr int kNodeTaken = 0x40000000;  // stack flag: a bucket whose test is passed
template <int W>
struct GroupWalkLds {
    static constexpr int kWide = W == 64 ? 16 * W : 8 * W;
    int stack[kWide + W + 96];
    int cand[W * (kTreeBucket + 1)];
};
using WaveWalkLds = GroupWalkLds<64>;

// The tree walk of one particle by W lanes (a power of two): the same visits as
// tree_walk (h_pair < 0: radius R only; else max(h_pair, node hmax)), handed out
// W slots at a time, f(slot, valid) called by the W lanes together.
//
// Walked alone, a node costs its load's full latency, and so does each step of
// the next: the few particles whose search sphere reaches into a dense clump
// (some 2,000 of 250,000 in a set of Plummer spheres) held a stage for
// milliseconds.  Here the lanes test the first W entries of a stack of pending
// nodes at once; a node that is opened leaves its two children in its place.
// ORDERED: slots leave in ascending order, so a bucket past an opened node waits
// on the stack.
// With budget > 0 the walk ends, returning false, once it has passed that many
// slots.
template <int W, bool ORDERED, typename F>
__device__ __forceinline__ bool group_tree_walk(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                                double h_pair, int lane, GroupWalkLds<W> &lds, F &&f, int budget = 0)
{
    int top = 0, fill = 0, passed = 0;
    if (G.root != kTreeEnd) {
        if (lane == 0) lds.stack[0] = G.root;
        top = 1;
    }
    wave_lds_fence();
    // a well-formed tree has 2 count - 1 nodes, and each turn takes at least one off
    for (int turns = 2 * G.count; top > 0 && turns > 0; turns--) {
        const int m = min(min(top, W), max(1, lds.kWide + W - top));
        const int item = lane < m ? lds.stack[top - 1 - lane] : kTreeEnd;
        int beg = 0, end = -1, left = 0, right = 0;
        bool open = false, range = false;
        if (lane < m) {
            if (item < 0) {
                beg = end = -item - 1;
                range = true;
            } else {
                const TreeNode nd = T.nodes[item & ~kNodeTaken];
                beg = nd.link.y;
                end = nd.link.z;
                left = nd.link.x;
                right = nd.link.w;
                bool in = true;
                if (!(item & kNodeTaken)) {
                    const double hm = nd.lo.w;
                    const double Rn = (h_pair < 0) ? R : ((hm > h_pair) ? hm : h_pair);
                    const double gx = periodic_gap(x[0], nd.lo.x, nd.hi.x, G.box.L[0]);
                    const double gy = periodic_gap(x[1], nd.lo.y, nd.hi.y, G.box.L[1]);
                    const double gz = periodic_gap(x[2], nd.lo.z, nd.hi.z, G.box.L[2]);
                    in = gx * gx + gy * gy + gz * gz <= Rn * Rn * (1.0 + 1e-9);
                }
                range = in && end - beg < kTreeBucket;
                open = in && !range;
            }
        }
        const uint64_t opened = group_ballot<W>(open);
        const int front = ORDERED && opened ? __ffsll((unsigned long long)opened) - 1 : W;
        const bool out = range && lane < front;
        const int n_slots = out ? end - beg + 1 : 0, n_push = open ? 2 : (range && !out ? 1 : 0);
        int sum = n_slots << 16 | n_push;
#pragma unroll
        for (int off = 1; off < W; off <<= 1) {
            const int o = __shfl_up(sum, off, W);
            if (lane >= off) sum += o;
        }
        const int total = __shfl(sum, W - 1, W);
        int c = fill + (sum >> 16) - n_slots;
        for (int j = beg; out && j <= end; j++) lds.cand[c++] = j;
        top += (total & 0xffff) - m;
        const int p = top - 1 - ((sum & 0xffff) - n_push);
        if (open) {
            lds.stack[p] = left;
            lds.stack[p - 1] = right;
        } else if (n_push) {
            lds.stack[p] = item < 0 ? item : item | kNodeTaken;
        }
        fill += total >> 16;
        passed += total >> 16;
        if (budget && passed > budget) return false;
        wave_lds_fence();
        if (fill >= W) {
            int done = 0;
            for (; fill - done >= W; done += W) walk_call(f, lds.cand[done + lane], true, false);
            fill -= done;
            const int rest = lds.cand[done + lane];
            wave_lds_fence();
            if (lane < fill) lds.cand[lane] = rest;
            wave_lds_fence();
        }
    }
    walk_call(f, lane < fill ? lds.cand[lane] : 0, lane < fill, true);
    wave_lds_fence();
    return true;
}

template <bool ORDERED, typename F>
__device__ __forceinline__ bool wave_tree_walk(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                               double h_pair, int lane, WaveWalkLds &lds, F &&f, int budget = 0)
{
    return group_tree_walk<64, ORDERED>(T, G, x, R, h_pair, lane, lds, f, budget);
}

// The same walk (radius R only, slots in no order) by a workgroup of WAVES
// wavefronts, for the walks over thousands of slots: stack and slots in common, so
// that the wavefronts stay alike busy.  A split of the stack among them, each
// going on alone, left most waiting for the one with the densest subtree.
template <int WAVES>
struct BlockWalkLds {
    static constexpr int kThreads = 64 * WAVES, kWide = 8 * kThreads;
    int stack[kWide + kThreads + 96];
    int cand[kThreads * (kTreeBucket + 1)];
    int total[WAVES];
};

template <int WAVES, typename F>
__device__ __forceinline__ void block_tree_walk(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                                BlockWalkLds<WAVES> &lds, F &&f)
{
    constexpr int kThreads = 64 * WAVES;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int top = G.root != kTreeEnd ? 1 : 0, fill = 0;
    if (tid == 0) lds.stack[0] = G.root;
    __syncthreads();
    for (int turns = 2 * G.count; top > 0 && turns > 0; turns--) {
        const int m = min(min(top, kThreads), max(1, lds.kWide + kThreads - top));
        const int item = tid < m ? lds.stack[top - 1 - tid] : kTreeEnd;
        int beg = 0, end = -1, left = 0, right = 0;
        bool open = false, range = false;
        if (tid < m) {
            if (item < 0) {
                beg = end = -item - 1;
                range = true;
            } else {
                const TreeNode nd = T.nodes[item];
                beg = nd.link.y;
                end = nd.link.z;
                left = nd.link.x;
                right = nd.link.w;
                const double gx = periodic_gap(x[0], nd.lo.x, nd.hi.x, G.box.L[0]);
                const double gy = periodic_gap(x[1], nd.lo.y, nd.hi.y, G.box.L[1]);
                const double gz = periodic_gap(x[2], nd.lo.z, nd.hi.z, G.box.L[2]);
                const bool in = gx * gx + gy * gy + gz * gz <= R * R * (1.0 + 1e-9);
                range = in && end - beg < kTreeBucket;
                open = in && !range;
            }
        }
        const int n_slots = range ? end - beg + 1 : 0, n_push = open ? 2 : 0;
        int sum = n_slots << 16 | n_push;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(sum, off, 64);
            if (lane >= off) sum += o;
        }
        if (lane == 63) lds.total[wave] = sum;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const int v = lds.total[w];
            if (w < wave) before += v;
            total += v;
        }
        sum += before;
        int c = fill + (sum >> 16) - n_slots;
        for (int j = beg; range && j <= end; j++) lds.cand[c++] = j;
        top += (total & 0xffff) - m;
        const int p = top - 1 - ((sum & 0xffff) - n_push);
        if (open) {
            lds.stack[p] = left;
            lds.stack[p - 1] = right;
        }
        fill += total >> 16;
        __syncthreads();
        if (fill >= kThreads) {
            int done = 0;
            for (; fill - done >= kThreads; done += kThreads) f(lds.cand[done + tid], true);
            fill -= done;
            const int rest = lds.cand[done + tid];
            __syncthreads();
            if (tid < fill) lds.cand[tid] = rest;
            __syncthreads();
        }
    }
    f(tid < fill ? lds.cand[tid] : 0, tid < fill);
    __syncthreads();
}

// Every candidate of one particle (search radius R around x), spread over the
// 64 lanes of a wavefront that walks the tree or the grid in step: each lane
// receives its share, f(k).  For the few particles whose search covers far
// more candidates than a lane can walk alone.  h_pair >= 0 (the pair search,
// R = max(h_i, box hsml max), h_pair = h_i): cells and nodes are also culled
// by the largest hsml they hold, as in the pair walks.
template <typename F>
__device__ __forceinline__ void wave_candidates(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                                int lane, WaveWalkLds &lds, F &&f, double h_pair = -1.0)
{
    if (T.nodes) {
        wave_tree_walk<false>(T, G, x, R, h_pair, lane, lds, [&](int j, bool valid) {
            if (valid) f(j);
        });
    } else {
        bool full[3];
        for_each_cell(G.grid, x, R, full, [&](int, int, int, int beg, int end) {
            for (int k = beg + lane; k < end; k += 64) f(k);
        }, h_pair);
    }
}

// Every grid candidate of one particle within R of x, spread over W lanes that
// walk the cells in step (`sub` = 0 .. W - 1): f(k) for each lane's share.  With
// budget > 0 the walk ends, returning false, once it has passed that many
// candidates (charged a cell at a time, so alike on every lane).
template <int W, typename F>
__device__ __forceinline__ bool group_candidates(const BoxDesc &G, const double x[3], double R, int sub, int budget,
                                                 F &&f)
{
    int visited = 0;
    bool full[3], ok = true;
    for_each_cell(G.grid, x, R, full, [&](int, int, int, int beg, int end) -> bool {
        visited += end - beg;
        if (budget && visited > budget) {
            ok = false;
            return false;
        }
        for (int k = beg + sub; k < end; k += W) f(k);
        return true;
    });
    return ok;
}

// The pairs of one particle (search radius R = max(h_i, box hsml max); cells and
// nodes culled by their hsml max against h_pair = h_i, as in the pair walks), by a
// wavefront: every candidate for which accept(j) is handed to eval(j), 64 at a
// time, one per lane, so that the lanes of the costly eval are full whatever
// share of the candidates the test leaves.  Grid: the pairs come in the order of
// the walk and pair k goes to lane k % 64, as it does from the pair list `row`
// of `n` entries (n < 0: none), which replaces the walk: sums do not depend on
// it.  (With an axis walked whole the list may be in another order; then the
// walk.)  The particles of 64 cells at a time are numbered through and tested 64 by
// 64, each once: full lanes whether a cell holds a particle or two or thousands.  (Whole
// cells to a lane, tested again for each 64 pairs taken, were quadratic in a dense
// cell: 32 k particles in Plummer spheres on the grid, force stage 231 ms against 1.0;
// 68,921 particles of 128 neighbours, all past their lists, 6.6 against 2.3.)
// FP64 redo of 756 k FP32 particles in shear layers: fluxes 0.085 ms against 0.64,
// gradients 0.061 against 0.157, with every candidate evaluated by the lane that
// found it.
struct WavePairLds {
    WaveWalkLds walk;
    int pair[128];
};

template <typename A, typename E>
__device__ __forceinline__ void wave_pairs(const TreeArgs &T, const BoxDesc &G, const double x[3], double R,
                                           double h_pair, int lane, const int *row, int n, WavePairLds &lds, A &&accept,
                                           E &&eval)
{
    int fill = 0;
    if (T.nodes) {
        wave_tree_walk<false>(T, G, x, R, h_pair, lane, lds.walk, [&](int j, bool valid, bool last) {
            const bool in = valid && accept(j);
            const uint64_t bits = __ballot(in);
            if (in) lds.pair[fill + __popcll(bits & ((1ull << lane) - 1))] = j;
            fill += __popcll(bits);
            wave_lds_fence();
            while (fill >= 64 || (last && fill > 0)) {
                if (lane < fill) eval(lds.pair[lane]);
                fill = max(fill - 64, 0);
                const int rest = lds.pair[64 + lane];
                wave_lds_fence();
                if (lane < fill) lds.pair[lane] = rest;
                wave_lds_fence();
            }
        });
        return;
    }
    const Grid &g = G.grid;
    int lo[3], nc[3];
    bool full[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        full[a] = !(R * g.inv_s[a] < 0.5 * g.nc[a] - 2.0);
        if (!full[a]) {
            lo[a] = (int)floor((x[a] - R) * g.inv_s[a] - 1e-6);
            nc[a] = (int)floor((x[a] + R) * g.inv_s[a] + 1e-6) - lo[a] + 1;
        } else {
            lo[a] = 0;
            nc[a] = g.nc[a];
        }
    }
    const double R2 = R * R * (1.0 + 1e-9);
    const double hp2 = h_pair * h_pair * (1.0 + 1e-9);
    const bool listed = n >= 0 && !(full[0] || full[1] || full[2]);
    const int n_cells = nc[0] * nc[1] * nc[2];
    // where the walk stands: the candidates of this turn's cells (candidate u of the
    // lane's cell, whose last is number upto - 1, is slot + u), `at` of `total` tested
    int next = 0, total = 0, at = 0, upto = 0, slot = 0;
    for (bool last = false; !last || fill > 0;) {
        if (listed) {
            fill = min(64, n - next);
            if (lane < fill) lds.pair[lane] = row[next + lane];
            next += 64;
            last = next >= n;
        }
        while (!listed && !last && fill < 64) {
            if (at >= total) {
                if (next >= n_cells) {
                    last = true;
                    break;
                }
                const int c = next + lane;
                next += 64;
                int2 slots = make_int2(0, 0);
                if (c < n_cells) {
                    const int cz = lo[2] + c % nc[2];
                    const int cy = lo[1] + (c / nc[2]) % nc[1];
                    const int cx = lo[0] + c / (nc[2] * nc[1]);
                    const int wx = (cx < 0) ? cx + g.nc[0] : ((cx >= g.nc[0]) ? cx - g.nc[0] : cx);
                    const int wy = (cy < 0) ? cy + g.nc[1] : ((cy >= g.nc[1]) ? cy - g.nc[1] : cy);
                    const int wz = (cz < 0) ? cz + g.nc[2] : ((cz >= g.nc[2]) ? cz - g.nc[2] : cz);
                    const double gx = full[0] ? 0.0 : axis_gap(x[0], cx * g.s[0], g.s[0]);
                    const double gy = full[1] ? 0.0 : axis_gap(x[1], cy * g.s[1], g.s[1]);
                    const double gz = full[2] ? 0.0 : axis_gap(x[2], cz * g.s[2], g.s[2]);
                    const double d2 = gx * gx + gy * gy + gz * gz;
                    const int cell = (wx * g.nc[1] + wy) * g.nc[2] + wz;
                    bool in = !(d2 > R2);
                    if (in && d2 > hp2) {
                        const double hm = g.hmax[cell];
                        in = !(d2 > hm * hm * (1.0 + 1e-9));
                    }
                    if (in) slots = g.range[cell];
                }
                const int size = slots.y - slots.x;
                upto = size;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const int o = __shfl_up(upto, off, 64);
                    if (lane >= off) upto += o;
                }
                slot = slots.x - (upto - size);
                total = __shfl(upto, 63, 64);
                at = 0;
                continue;
            }
            const int u = at + lane;
            int cell = 0;  // the first whose last candidate is not before u
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (__shfl(upto, cell + step - 1, 64) <= u) cell += step;
            const int j = __shfl(slot, cell, 64) + u;
            const bool in = u < total && accept(j);
            const uint64_t bits = __ballot(in);
            if (in) lds.pair[fill + __popcll(bits & ((1ull << lane) - 1))] = j;
            fill += __popcll(bits);
            at += 64;
        }
        wave_lds_fence();
        if (lane < fill) eval(lds.pair[lane]);
        fill = max(fill - 64, 0);
        wave_lds_fence();
        if (fill > 0) {
            const int rest = lds.pair[64 + lane];
            wave_lds_fence();
            if (lane < fill) lds.pair[lane] = rest;
            wave_lds_fence();
        }
    }
}

// sum over the G lanes of one particle (every lane gets the result)
template <int G>
__device__ __forceinline__ double group_sum(double v)
{
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <int G>
__device__ __forceinline__ double group_max(double v)
{
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o > v) ? o : v;
    }
    return v;
}

template <int G>
__device__ __forceinline__ double group_min(double v)
{
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o < v) ? o : v;
    }
    return v;
}

template <int G>
__device__ __forceinline__ int group_sum_int(int v)
{
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// bitwise or over the G lanes of one particle
template <int G>
__device__ __forceinline__ uint64_t group_or(uint64_t v)
{
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) v |= __shfl_xor((unsigned long long)v, off, 64);
    return v;
}

// The pair lists of 64 / kForceLanes particles, one wavefront (a workgroup of its
// own), kForceLanes lanes per particle: step by step each lane takes one pair,
// visit(own, other, x_j, j, k) with both records in LDS.
//
// A lane that reads its neighbour's record itself costs the address unit one
// cycle per lane and 16 bytes (20 loads of 64 lanes: 1,280 cycles a step for the
// FP64 record, more than the 1,000 of the arithmetic on a CU's four SIMDs).
// Four lanes reading 64 adjacent bytes cost one, so the wavefront fetches the 64
// records of a step together and passes them on through LDS; the loads of the
// next step are in flight while this one computes.  Eight lanes per particle
// instead of one keep the neighbours of all particles in flight on an XCD within
// its 4 MB L2 (L2 misses 5,150 against 318 lines per 64 particles of a 2.1 M set)
// and let them share i's record in LDS instead of each holding it in registers.
template <typename REC>
struct PairLoopLds {
    REC other[64];
    REC own[64 / kForceLanes];
};

template <typename REC, typename F>
__device__ __forceinline__ void pair_list_loop(PairLoopLds<REC> &lds, const REC *__restrict__ rec,
                                               const double4 *__restrict__ posm, const int *row, int n, int i,
                                               F &&visit)
{
    constexpr int kChunks = (int)(sizeof(REC) / 16), kSegments = kChunks / 4, kRest = kChunks % 4;
    static_assert(sizeof(REC) % 16 == 0, "records of whole 16-byte chunks");
    using Chunk = double __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, sub = lane % kForceLanes, g = lane / kForceLanes;
    int steps = (n + kForceLanes - 1) / kForceLanes;
    for (int off = 32; off >= kForceLanes; off >>= 1) steps = max(steps, __shfl_xor(steps, off, 64));
    // i's record
    {
        const double *src = reinterpret_cast<const double *>(rec + i);
        double *dst = reinterpret_cast<double *>(lds.own + g);
        for (int w = sub; w < (int)(sizeof(REC) / 8); w += kForceLanes) dst[w] = src[w];
    }
    Chunk seg[4][kSegments], rest[kRest > 0 ? kRest : 1];
    double4 xj;
    auto fetch = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const Chunk *src = reinterpret_cast<const Chunk *>(rec + __shfl(j, 16 * q + (lane >> 2), 64));
#pragma unroll
            for (int m = 0; m < kSegments; m++) seg[q][m] = src[4 * m + (lane & 3)];
        }
        const Chunk *src = reinterpret_cast<const Chunk *>(rec + j);
#pragma unroll
        for (int m = 0; m < kRest; m++) rest[m] = src[4 * kSegments + m];
        xj = posm[j];
    };
    // lanes past their list fetch i itself
    int j = sub < n ? row[sub] : i;
    int j_next = sub + kForceLanes < n ? row[sub + kForceLanes] : i;
    if (steps > 0) fetch(j);
    for (int it = 0; it < steps; it++) {
        wave_lds_fence();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            Chunk *dst = reinterpret_cast<Chunk *>(lds.other + 16 * q + (lane >> 2));
#pragma unroll
            for (int m = 0; m < kSegments; m++) dst[4 * m + (lane & 3)] = seg[q][m];
        }
        Chunk *dst = reinterpret_cast<Chunk *>(lds.other + lane);
#pragma unroll
        for (int m = 0; m < kRest; m++) dst[4 * kSegments + m] = rest[m];
        wave_lds_fence();
        const int k = it * kForceLanes + sub, j_now = j;
        const double4 x_now = xj;
        if (it + 1 < steps) {
            j = j_next;
            fetch(j);
            const int k2 = k + 2 * kForceLanes;
            j_next = k2 < n ? row[k2] : i;
        }
        if (k < n) visit(lds.own[g], lds.other[lane], x_now, j_now, k);
    }
}

// Whether the candidate row of radius^2 r2 around x holds the whole pair set
// {j : r < h_i or r < h_j}: no particle beyond the radius has an hsml that
// reaches x.  The box's largest hsml answers for most sets; else the cells in
// its reach do, each by its own largest.
__device__ __forceinline__ bool row_holds_pairs(const BoxDesc &B, const double x[3], double h_i, double r2)
{
    if (!(h_i * h_i <= r2)) return false;
    if (B.hmax * B.hmax <= r2) return true;
    const Grid &g = B.grid;
    bool full[3], holds = true;
    for_each_cell(g, x, B.hmax, full, [&](int cx, int cy, int cz, int beg, int end) -> bool {
        if (beg == end) return true;
        const int wx = (cx < 0) ? cx + g.nc[0] : ((cx >= g.nc[0]) ? cx - g.nc[0] : cx);
        const int wy = (cy < 0) ? cy + g.nc[1] : ((cy >= g.nc[1]) ? cy - g.nc[1] : cy);
        const int wz = (cz < 0) ? cz + g.nc[2] : ((cz >= g.nc[2]) ? cz - g.nc[2] : cz);
        const double hm = g.hmax[(wx * g.nc[1] + wy) * g.nc[2] + wz], hm2 = hm * hm * (1.0 + 1e-9);
        if (hm2 <= r2) return true;
        const double gx = full[0] ? 0.0 : axis_gap(x[0], cx * g.s[0], g.s[0]);
        const double gy = full[1] ? 0.0 : axis_gap(x[1], cy * g.s[1], g.s[1]);
        const double gz = full[2] ? 0.0 : axis_gap(x[2], cz * g.s[2], g.s[2]);
        holds = gx * gx + gy * gy + gz * gz > hm2;
        return holds;
    });
    return holds;
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ double wave_max(double v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o > v) ? o : v;
    }
    return v;
}

__device__ __forceinline__ double wave_min(double v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o < v) ? o : v;
    }
    return v;
}

// Run f(desc) for this lane's particle with its box descriptor, one
// wave-uniform box at a time: the box index is taken from the first lane still
// to run (readfirstlane), so the descriptor's fields are uniform and a
// wavefront that straddles two boxes runs the body twice with the lanes of
// each box.
template <typename F>
__device__ __forceinline__ void for_box(const BoxDesc *__restrict__ boxes, const int *box_of, int i, bool valid,
                                        F &&f)
{
    bool todo = valid;
    const int my_b = valid ? box_of[i] : 0;
    while (todo) {
        const int b = __builtin_amdgcn_readfirstlane(my_b);
        if (my_b == b) {
            f(boxes[b]);
            todo = false;
        }
    }
}

// hydro_final_operations_and_cleanup (hydro_toplevel.c:738-764) on the raw
// sums of one particle: dE -= v . a before the mass division
__device__ __forceinline__ void force_final_ops(double acc[3], double &dte, const double v[3], double m_i,
                                                double h_i, double max_hsml)
{
    dte -= (v[0] / 1.0) * acc[0];
    acc[0] /= m_i;
    dte -= (v[1] / 1.0) * acc[1];
    acc[1] /= m_i;
    dte -= (v[2] / 1.0) * acc[2];
    acc[2] /= m_i;
    dte /= m_i;
    if (h_i >= 0.99 * max_hsml) dte = 0;
}

// The sums of the list kernels' kForceLanes lanes kept by one lane for the forms
// without them, added up in their order (group_sum's), so that all forms give the
// same bits.  In LDS, part_bytes(threads) of it: an array indexed by the pair's
// number lies in scratch memory, 256 bytes a lane.
struct LaneSums {
    double *at;  // [lane][component][thread]
    int stride;
    __device__ __forceinline__ LaneSums(double *lds) : at(lds + threadIdx.x), stride((int)blockDim.x)
    {
#pragma unroll
        for (int k = 0; k < 4 * kForceLanes; k++) at[k * stride] = 0;
    }
    __device__ __forceinline__ void add(int lane, const double v[4])
    {
#pragma unroll
        for (int c = 0; c < 4; c++) at[(4 * lane + c) * stride] += v[c];
    }
    __device__ __forceinline__ void fold()
    {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            double v[kForceLanes];
#pragma unroll
            for (int l = 0; l < kForceLanes; l++) v[l] = at[(4 * l + c) * stride];
#pragma unroll
            for (int off = kForceLanes / 2; off > 0; off >>= 1)
#pragma unroll
                for (int l = 0; l < off; l++) v[l] += v[l + off];
            at[c * stride] = v[0];
        }
    }
    __device__ __forceinline__ double total(int c) const { return at[c * stride]; }
};
// one sum, with the same face
struct OwnSums {
    double v[4] = {0, 0, 0, 0};
    __device__ __forceinline__ OwnSums(double *) {}
    __device__ __forceinline__ void add(int, const double x[4])
    {
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] += x[c];
    }
    __device__ __forceinline__ double total(int c) const { return v[c]; }
};
inline size_t part_bytes(unsigned threads) { return sizeof(double) * 4 * kForceLanes * threads; }

// this workgroup's copy of a stage's counters
__device__ __forceinline__ Counters *ctr_slot(Counters *c) { return c + (blockIdx.x & (kCtrSpread - 1)); }

// wavefront-wide sum, then one atomic per wavefront
__device__ __forceinline__ void wave_add_u64(unsigned long long *dst, unsigned long long v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(dst, v);
}

// MINMAX_CHECK of the reference (else-if: a new minimum is not also tested
// as a maximum, gradients.c:29).  Written with selects: as two conditional
// stores the compiler may merge them into one store through a selected
// address, which moves the accumulators to scratch memory.
template <typename T>
__device__ __forceinline__ void minmax_check(T x, T &mn, T &mx)
{
    const bool lt = x < mn;
    const bool gt = !lt && (x > mx);
    mn = lt ? x : mn;
    mx = gt ? x : mx;
}

// LDS of one wavefront for index rows: kListChunk entries per lane, entry c of
// lane l at [c * 64 + l], so that same-c accesses hit distinct banks.
constexpr int kWaveChunk = kListChunk * 64;

__device__ __forceinline__ int *wave_chunk(int *lds) { return lds + (threadIdx.x >> 6) * kWaveChunk; }

// One lane's staged chunk -> 64 bytes of its row.
__device__ __forceinline__ void flush_list_chunk(const int *chunk, int *dst)
{
    const int *c = chunk + (threadIdx.x & 63);
    int4 *d = reinterpret_cast<int4 *>(dst);
#pragma unroll
    for (int q = 0; q < kListChunk / 4; q++)
        d[q] = make_int4(c[(4 * q + 0) * 64], c[(4 * q + 1) * 64], c[(4 * q + 2) * 64], c[(4 * q + 3) * 64]);
}

// 64 bytes of a lane's row -> its chunk.  Read entry by entry as the loop goes,
// the row's line is out of the 32 KB L1 again before the next entry (64 rows of
// a wavefront are 64 lines).
__device__ __forceinline__ void load_list_chunk(int *chunk, const int *src)
{
    int *c = chunk + (threadIdx.x & 63);
    const int4 *q4 = reinterpret_cast<const int4 *>(src);
#pragma unroll
    for (int q = 0; q < kListChunk / 4; q++) {
        const int4 v = q4[q];
        c[(4 * q + 0) * 64] = v.x;
        c[(4 * q + 1) * 64] = v.y;
        c[(4 * q + 2) * 64] = v.z;
        c[(4 * q + 3) * 64] = v.w;
    }
}

// f(entry) for the n entries of a lane's row, in order, through its chunk
// (a row's memory is whole chunks).
template <typename F>
__device__ __forceinline__ void for_row(int *chunk, const int *row, int n, F &&f)
{
    const int *c = chunk + (threadIdx.x & 63);
    for (int k = 0; k < n; k += kListChunk) {
        load_list_chunk(chunk, row + k);
        const int m = min(kListChunk, n - k);
        for (int e = 0; e < m; e++) f(c[e * 64]);
    }
}

// f(entry a, entry b, whether b counts) two at a time, for loads in flight
template <typename F>
__device__ __forceinline__ void for_row_pairs(int *chunk, const int *row, int n, F &&f)
{
    const int *c = chunk + (threadIdx.x & 63);
    for (int k = 0; k < n; k += kListChunk) {
        load_list_chunk(chunk, row + k);
        const int m = min(kListChunk, n - k);
        for (int e = 0; e < m; e += 2) {
            const bool second = e + 1 < m;
            const int j = c[e * 64];
            f(j, second ? c[(e + 1) * 64] : j, second);
        }
    }
}

// Store N 8-byte words of each lane's record i (stride in words, from base)
// through the wavefront's LDS (1024 ints): eight lanes write 64 adjacent bytes of
// one record.  A lane's own stores of a record go out as one request per lane
// and 8 or 16 bytes (2,364 requests per wavefront of the gradient kernel).
// Called by all 64 lanes; `valid` lanes store.
template <int N>
__device__ __forceinline__ void wave_store_records(int *lds, double *base, size_t stride, int i, bool valid,
                                                   const double (&w)[N])
{
    double *buf = reinterpret_cast<double *>(lds);
    const int lane = threadIdx.x & 63, word = lane & 7;
#pragma unroll
    for (int p = 0; p < N; p += 8) {
        wave_lds_fence();
#pragma unroll
        for (int c = 0; c < 8; c++)
            if (p + c < N) buf[lane * 8 + (c ^ word)] = w[p + c];
        wave_lds_fence();
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int l = it * 8 + (lane >> 3);  // whose record
            const int il = __shfl(i, l, 64);
            const bool ok = __shfl((int)valid, l, 64) != 0;
            const double v = buf[l * 8 + (word ^ (l & 7))];
            if (ok && p + word < N) base[(size_t)il * stride + p + word] = v;
        }
    }
}

}  // namespace gzm
