// gzm_density.hip -- the density stage of the FP64 hsml iteration (precisions
// 0 and 1; also the FP64 redo of precision 2) for gfx950.
//
// A particle's iteration reads only its own sums, so no sweep has to be a
// launch of its own and nothing is compacted or counted on the host between
// sweeps.  The kernels of a stage:
//
//   density_rows_kernel   candidates of every active particle within
//                         kDensityCacheFactor * hsml, in walk order (a pure
//                         distance filter over the grid or tree)
//   density_stage_kernel  the first two sweeps over the rows, a launch each
//                         (nearly every particle of an even set needs exactly two)
//   density_more_kernel   what is left by then, packed anew for every sweep (not
//                         for few particles in the grid)
//   density_tail_kernel   the last of those: 16 lanes each, iterating to convergence
//   density_far_kernel    of those, the particles whose walk passes the candidate
//                         budget; for few particles all that is left: a wavefront
//                         each, iterating to convergence
//
// The tree has kernels of its own for the particles that have to walk.
//
// The lists between them live on the device.
//
// 128^3 blast (2.1 M particles, 33 pairs and 1.97 sweeps each): rows 0.86, sweeps
// 0.66 + 0.66, tail and far 0.03 ms; the launch per sweep with its walk that this
// replaces took 2 x 1.41 ms and a host round trip per sweep.  32^3 lattice: rows
// 0.033, sweeps 2 x 0.024 ms (2 x 0.11 ms).  Bound by the latency of the
// candidate loads (45 % VALU busy, 500 cycles per load at 5 waves per SIMD).
#include "grid_device.h"
#include "gzm_internal.h"

namespace gzm {

namespace {

constexpr int kTailLanes = 16;
constexpr int kFarWaves = 4;
constexpr int kNoRow = kDensityCacheCap + 1;
constexpr int kWideRow = kNoRow + 1;  // row_n where the walk for the row passed its candidate budgets
// iter of a particle whose iteration has ended; beside the sweeps done, of one that is in
// the tail list
constexpr int kDone = -1, kListed = 1 << 30;

// sums of one candidate already known to lie within h (density.c:252-347).
// MFV: also m_j W_ij v_j into pv (density.c:291-293 for r = 0, 331-334 as
// v_i - (v_i - v_j) otherwise), the sum behind ParticleVel.
template <bool MFV>
__device__ __forceinline__ void density_add(const double dp[3], double r2, double m_j, const double4 &vi,
                                            const double4 &vj, double hinv, double hinv3, double hinv4,
                                            DensitySums &S, double *pv)
{
    const double r = sqrt(r2);
    const double u = r * hinv;
    double wk, dwk;
    kernel_wdw(u, hinv3, hinv4, wk, dwk);
    S.ngb += wk;
    S.rho += m_j * wk;
    S.dhsml += -(3 * hinv * wk + u * dwk);
    if (r > 0) {
        S.t00 += wk * dp[0] * dp[0];
        S.t01 += wk * dp[0] * dp[1];
        S.t02 += wk * dp[0] * dp[2];
        S.t11 += wk * dp[1] * dp[1];
        S.t12 += wk * dp[1] * dp[2];
        S.t22 += wk * dp[2] * dp[2];
        S.f0 += wk * dp[0];
        S.f1 += wk * dp[1];
        S.f2 += wk * dp[2];
        const double dv0 = vi.x - vj.x, dv1 = vi.y - vj.y, dv2 = vi.z - vj.z;
        if (MFV) {
            const double mj_wk = m_j * wk;
            pv[0] += mj_wk * (vi.x - dv0);
            pv[1] += mj_wk * (vi.y - dv1);
            pv[2] += mj_wk * (vi.z - dv2);
        }
        S.divvel -= dwk * (dp[0] * dv0 + dp[1] * dv1 + dp[2] * dv2) / r;
    } else if (MFV) {
        const double mj_wk = m_j * wk;
        pv[0] += mj_wk * vj.x;
        pv[1] += mj_wk * vj.y;
        pv[2] += mj_wk * vj.z;
    }
}

template <int G, bool MFV>
__device__ __forceinline__ void group_sums(DensitySums &S, double *pv)
{
    S.ngb = group_sum<G>(S.ngb); S.rho = group_sum<G>(S.rho); S.dhsml = group_sum<G>(S.dhsml);
    S.divvel = group_sum<G>(S.divvel);
    S.t00 = group_sum<G>(S.t00); S.t01 = group_sum<G>(S.t01); S.t02 = group_sum<G>(S.t02);
    S.t11 = group_sum<G>(S.t11); S.t12 = group_sum<G>(S.t12); S.t22 = group_sum<G>(S.t22);
    S.f0 = group_sum<G>(S.f0); S.f1 = group_sum<G>(S.f1); S.f2 = group_sum<G>(S.f2);
    if (MFV) {
        pv[0] = group_sum<G>(pv[0]);
        pv[1] = group_sum<G>(pv[1]);
        pv[2] = group_sum<G>(pv[2]);
    }
}

// sums of a workgroup's wavefronts (each with its own in every lane), in their
// order, to all of them
template <int WAVES, bool MFV>
__device__ __forceinline__ void block_sums(DensitySums &S, double *pv)
{
    constexpr int kSums = MFV ? 16 : 13;
    __shared__ double lds[WAVES][16];
    double v[16] = {S.ngb, S.rho, S.dhsml, S.divvel, S.t00, S.t01, S.t02, S.t11, S.t12, S.t22, S.f0, S.f1, S.f2,
                    pv[0], pv[1], pv[2]};
    if (threadIdx.x % 64 == 0)
        for (int k = 0; k < kSums; k++) lds[threadIdx.x / 64][k] = v[k];
    __syncthreads();
    for (int k = 0; k < kSums; k++) {
        v[k] = lds[0][k];
        for (int w = 1; w < WAVES; w++) v[k] += lds[w][k];
    }
    __syncthreads();
    S.ngb = v[0]; S.rho = v[1]; S.dhsml = v[2]; S.divvel = v[3];
    S.t00 = v[4]; S.t01 = v[5]; S.t02 = v[6]; S.t11 = v[7]; S.t12 = v[8]; S.t22 = v[9];
    S.f0 = v[10]; S.f1 = v[11]; S.f2 = v[12];
    if (MFV) {
        pv[0] = v[13];
        pv[1] = v[14];
        pv[2] = v[15];
    }
}

// where one particle stands in its iteration
struct Iterate {
    double h, left, right, cn;
    int iter;
};

// One hsml step from the sums of sweep s.iter; true: sweep again.  On the
// last sweep (converged, a bracket failure, or the sweep limit) `write` stores
// the outputs with the final operations of density.c:880-1031.
__device__ __forceinline__ bool density_step(const DensityStageArgs &a, int i, bool write, const DensitySums &S,
                                             const double *pv, Iterate &s)
{
    DensityResult R;
    HsmlParams hp = a.hp;
    hp.iter = s.iter;
    const int res = hsml_update(hp, S, s.h, s.left, s.right, s.cn, R);
    s.cn = R.cn_stored;
    s.iter++;
    const bool again = (res == 1) && (s.iter <= a.maxiter);
    if (again || !write) return again;
    if (res != 0) atomicMax(&ctr_slot(a.ctr)->status, res < 0 ? 6 : 1155);
    a.hsml[i] = s.h;
    a.cn[i] = s.cn;
    a.dhsml[i] = R.dhsml;
    a.divvel[i] = R.divvel;
    a.fce[i] = R.fce;
    double2 *t2 = reinterpret_cast<double2 *>(a.nvt + 6 * (size_t)i);
#pragma unroll
    for (int k = 0; k < 3; k++) t2[k] = make_double2(R.nvt[2 * k], R.nvt[2 * k + 1]);
    const double4 vi = a.velu[i];
    if (a.pvel) {
        // MFV mesh motion 5 (density.c:886-894): 0.7 VelPred + 0.3 the kernel-weighted mean velocity
        const double eps_pvel = 0.3, d_sum = R.rho_sum;
        const double vv[3] = {vi.x, vi.y, vi.z};
        for (int k = 0; k < 3; k++)
            a.pvel[3 * (size_t)i + k] = (d_sum > 0) ? (1. - eps_pvel) * vv[k] + eps_pvel * pv[k] / d_sum : pv[k];
    }
    const double h = s.h, nn = R.num_ngb, m = a.posm[i].w;
    double d;
    // density.c:967-978 (MFM: own mass times the kernel number density)
    if ((h > 0) && (nn > 0)) d = m * nn / (kNormCoeff * cube(h));
    else if (h <= 0) d = 0;
    else d = m / (kNormCoeff * cube(h));
    a.rho[i] = d;
    a.pres[i] = a.gm1 * vi.w * d;                       // eos.c:58-61
    a.num_ngb[i] = (nn > 0) ? cbrt(nn) : 0;  // density.c:1020
    return again;
}

// leave particle i to the next sweep, or to the kernel that works through `list`
__device__ __forceinline__ void hand_on(const DensityStageArgs &a, int i, const Iterate &s, int *list, int *count)
{
    a.hsml[i] = s.h;
    a.left[i] = s.left;
    a.right[i] = s.right;
    a.cn[i] = s.cn;
    a.iter[i] = s.iter;
    if (list) list[atomicAdd(count, 1)] = i;
}

__device__ __forceinline__ Iterate take_up(const DensityStageArgs &a, int i)
{
    return {a.hsml[i], a.left[i], a.right[i], a.cn[i], a.iter[i] & ~kListed};
}

__device__ __forceinline__ void count_sweeps(const DensityStageArgs &a, unsigned long long pairs,
                                             unsigned long long sweeps, int max_iter)
{
    wave_add_u64(&ctr_slot(a.ctr)->interactions, pairs);
    wave_add_u64(&ctr_slot(a.ctr)->updates, sweeps);
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(max_iter, off, 64);
        max_iter = o > max_iter ? o : max_iter;
    }
    if ((threadIdx.x & 63) == 0 && max_iter > 0) atomicMax(&ctr_slot(a.ctr)->sweeps, max_iter);
}

// Candidate rows.  The walk tests every particle of the cells (nodes) that the
// radius touches, some 250 for 32 neighbours; testing only distances here and
// summing over the ~55 row entries afterwards keeps the lanes of the sums
// together (in one loop nearly every candidate step of a wavefront runs the
// pair body for the few lanes that have a neighbour there).  G = 1: one lane
// per particle, entries staged in LDS and stored as whole 64-byte chunks.
// Bound by VALU issue and the address unit alike (70 %, 69 % busy); the cells of a
// z column come from the sphere's width there, not from a test of each (3.55 M
// particles at half-hsml cells 1.98 -> 1.72 ms, 0.96 M at hsml cells 0.65 -> 0.58).
// G > 1 (few particles): each of the G lanes walks a z column of cells, same order
// (4,096 particles: 18 us, 32 k: 33 us; with the lanes sharing the candidates of one
// cell after the other, waiting for each cell's slots, 28 and 38 us); a column with
// more hits than a lane keeps sends its particle to that form.
// Returns the number of entries as stored in row_n, kNoRow or kWideRow where there is no row.
__device__ __forceinline__ double grid_row_r2(double h)
{
    const double Rc = kDensityCacheFactorGrid * h;
    return Rc * Rc;
}
// Whether to build a particle's row (of n_row entries in the radius^2 r2 tried last)
// anew for hsml h: it left the row, or there was none and it is now so much smaller that
// half the entries are left.
__device__ __forceinline__ bool row_wanted(int n_row, double r2, double h)
{
    return n_row <= kDensityCacheCap ? h * h > r2 : grid_row_r2(h) < 0.64 * r2;
}
// whether a walk of radius h passes more cells than one lane should
__device__ __forceinline__ bool many_cells(const Grid &g, double h)
{
    double cells = 1;
#pragma unroll
    for (int ax = 0; ax < 3; ax++) cells *= fmin((double)g.nc[ax], 2 * h * g.inv_s[ax] + 1);
    return cells > 512;
}
template <int G>
constexpr int kRowLds = G == 1 ? kListChunk * kBlock : kColumnHits * kBlock;
template <int G>
__device__ __forceinline__ int grid_row(const DensityStageArgs &a, const BoxDesc &B, int i, const double4 &pi, double h,
                                        int sub, int *lds, int budgets = 2)
{
    int *stage = wave_chunk(lds), *kept = lds;
    const double Rc = kDensityCacheFactorGrid * h;
    const double xs[3] = {pi.x, pi.y, pi.z};
    constexpr int cap = kDensityCacheCap;
    int *row = a.row_idx + (size_t)i * cap;
    // a row past its cap is of no use, so its walk ends there; a number of candidate
    // budgets bounds the walk where cells hold many more particles than neighbours
    const int limit = a.budget ? budgets * a.budget : 0x7fffffff;
    int m = 0, visited = 0;
    auto append = [&](int j, bool in) {
        if constexpr (G == 1) {
            if (!in) return;
            if (m < cap) {
                const int c = m & (kListChunk - 1);
                stage[c * 64 + (threadIdx.x & 63)] = j;
                if (c == kListChunk - 1) flush_list_chunk(stage, row + (m - c));
            }
            m++;
        } else {
            const uint64_t bits = group_ballot<G>(in);
            const int k = m + __popcll(bits & ((1ull << sub) - 1));
            if (in && k < cap) row[k] = j;
            m += __popcll(bits);
        }
    };
    // FP32 distances with a margin for their rounding (2^-24 of a side per
    // coordinate): the row may hold a few more than the exact radius
    // asks for, never fewer, and a candidate is one 16-byte load.  In units
    // of the box: the squares of a galaxy's centimetres overflow FP32.
    const float Lx = (float)(B.box.L[0] * B.unit), Ly = (float)(B.box.L[1] * B.unit), Lz = (float)(B.box.L[2] * B.unit);
    const float Rf = (float)(Rc * B.unit) * (1 + 1e-6f) + 5e-7f * fmaxf(Lx, fmaxf(Ly, Lz));
    const float Rf2 = Rf * Rf * (1 + 1e-6f);
    const float4 fi = a.posf[i];
    // the image of cell (cx, cy, cz) that the walk reached is the nearest one
    // wherever the axis is not walked whole
    auto near = [&](const float4 &pj, bool whole, int cx, int cy, int cz) {
        const float ox = fi.x - (cx < 0 ? -Lx : (cx >= B.grid.nc[0] ? Lx : 0.0f));
        const float oy = fi.y - (cy < 0 ? -Ly : (cy >= B.grid.nc[1] ? Ly : 0.0f));
        const float oz = fi.z - (cz < 0 ? -Lz : (cz >= B.grid.nc[2] ? Lz : 0.0f));
        float dx = ox - pj.x, dy = oy - pj.y, dz = oz - pj.z;
        if (whole) {
            dx -= Lx * rintf(dx / Lx);
            dy -= Ly * rintf(dy / Ly);
            dz -= Lz * rintf(dz / Lz);
        }
        return dx * dx + dy * dy + dz * dz < Rf2 && pj.w > 0;
    };
    auto run = [&](const bool full[3], int cx, int cy, int cz, int beg, int end) -> bool {
        visited += end - beg;
        if (visited > limit) return false;
        const bool whole = full[0] || full[1] || full[2];
        // two candidates in flight: the walk waits on these loads
        constexpr int U = 2;
        for (int k = beg + sub; k - sub < end; k += U * G) {
            float4 p[U];
#pragma unroll
            for (int c = 0; c < U; c++) p[c] = a.posf[min(k + c * G, end - 1)];
#pragma unroll
            for (int c = 0; c < U; c++)
                if (G > 1 || c == 0 || k + c < end) append(k + c * G, k + c * G < end && near(p[c], whole, cx, cy, cz));
        }
        return m <= cap;
    };
    bool listed = false;
    if constexpr (G > 1) {
        // (a column with that many candidates is better shared by many lanes)
        m = for_columns<G>(B.grid, xs, Rc, sub, G > 8 ? min(limit, 4 * kColumnHits) : limit, kept + threadIdx.x,
                           [&](int j, bool whole, int cx, int cy, int cz) {
            return near(a.posf[j], whole, cx, cy, cz);
        }, [&](int k, int j) {
            if (k < cap) row[k] = j;
        });
        listed = m >= 0;
        if (!listed) m = 0;
    }
    if (!listed) for_each_run(B.grid, xs, Rc, run);
    if (visited > limit) m = kWideRow;
    if (G == 1 && m < cap && (m & (kListChunk - 1)))
        flush_list_chunk(stage, row + (m & ~(kListChunk - 1)));
    if (m > cap && m != kWideRow) m = kNoRow;
    if (sub == 0) {
        a.row_n[i] = m;
        a.row_r2[i] = grid_row_r2(h);
    }
    return m;
}

template <int G>
__global__ __launch_bounds__(kBlock) void density_rows_kernel(DensityStageArgs a)
{
    __shared__ __align__(16) int lds[kRowLds<G>];
    const int gt = xcd_block() * kBlock + (int)threadIdx.x;
    const int t = gt / G, sub = gt % G;
    const bool valid = t < a.n_active;
    for_box(a.boxes, a.box_of, valid ? a.active[t] : 0, valid, [&](const BoxDesc &B) {
        const int i = a.active[t];
        const double4 pi = a.posm[i];
        if (!(pi.w > 0)) {  // density_isactive: gas with mass > 0 (density.c:85)
            if (sub == 0) a.row_n[i] = kNoRow;
            return;
        }
        double h = a.hsml[i];
        if ((h < 0) || !isfinite(h) || (h > 0.99 * a.hp.max_hsml)) {  // density.c:484
            h = 0.99 * a.hp.max_hsml;
            if (sub == 0) a.hsml[i] = h;
        }
        grid_row<G>(a, B, i, pi, h, sub, lds);
    });
}

// Candidate rows of the tree, kRowLanes lanes per particle (group_tree_walk).  With
// one lane each the longest walks of a wavefront's lanes set its time, node after
// node at the latency of each load: 1.15 ms for 250 k particles in Plummer spheres,
// now 0.63
// (16 lanes 0.69, 4 lanes 1.01).
constexpr int kRowLanes = 8;
__global__ __launch_bounds__(kBlock) void density_tree_rows_kernel(DensityStageArgs a)
{
    __shared__ GroupWalkLds<kRowLanes> walk[kBlock / kRowLanes];
    const int gt = xcd_block() * kBlock + (int)threadIdx.x;
    const int t = gt / kRowLanes, sub = gt % kRowLanes;
    const bool valid = t < a.n_active;
    for_box(a.boxes, a.box_of, valid ? a.active[t] : 0, valid, [&](const BoxDesc &B) {
        const int i = a.active[t];
        const double4 pi = a.posm[i];
        if (!(pi.w > 0)) {  // density_isactive: gas with mass > 0 (density.c:85)
            if (sub == 0) a.row_n[i] = kNoRow;
            return;
        }
        double h = a.hsml[i];
        if ((h < 0) || !isfinite(h) || (h > 0.99 * a.hp.max_hsml)) {  // density.c:484
            h = 0.99 * a.hp.max_hsml;
            if (sub == 0) a.hsml[i] = h;
        }
        const double Rc = kDensityCacheFactor * h, Rc2 = Rc * Rc;
        const double xs[3] = {pi.x, pi.y, pi.z};
        int *row = a.row_idx + (size_t)i * kDensityCacheCap;
        int m = 0;
        const bool whole = group_tree_walk<kRowLanes, true>(a.tree, B, xs, Rc, -1.0, sub, walk[threadIdx.x / kRowLanes],
                                                            [&](int j, bool in) {
            if (in) {
                const double4 pj = a.posm[j];
                double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
                wrap_dp(B.box, dp);
                const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                in = r2 < Rc2 && pj.w > 0;
            }
            const uint64_t bits = group_ballot<kRowLanes>(in);
            const int k = m + __popcll(bits & ((1ull << sub) - 1));
            if (in && k < kDensityCacheCap) row[k] = j;
            m += __popcll(bits);
        }, a.budget ? 2 * a.budget : 0);
        if (sub == 0) {
            a.row_n[i] = whole && m <= kDensityCacheCap ? m : kNoRow;
            a.row_r2[i] = Rc2;
        }
    });
}

// One sweep of a particle over its row, G lanes; true: sweep again.
template <bool MFV, int G>
__device__ __forceinline__ bool row_sweep(const DensityStageArgs &a, const BoxDesc &B, int i, const double4 &pi, int n,
                                          int sub, int *chunk, Iterate &s, unsigned long long &cnt)
{
    const double4 vi = a.velu[i];
    const int *row = a.row_idx + (size_t)i * kDensityCacheCap;
    const double h2 = s.h * s.h;
    double hinv, hinv3, hinv4;
    kernel_hinv(s.h, hinv, hinv3, hinv4);
    DensitySums S = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double pv[3] = {0, 0, 0};
    auto pair = [&](auto near, int j, const double4 &pj) {
        double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
        if constexpr (near.value) wrap_near(B.box, dp);
        else wrap_dp(B.box, dp);
        const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
        if (!(r2 < h2)) return;
        cnt++;
        density_add<MFV>(dp, r2, pj.w, vi, a.velu[j], hinv, hinv3, hinv4, S, pv);
    };
    auto scan = [&](auto near) {
        if constexpr (G == 1) {
            for_row_pairs(chunk, row, n, [&](int j0, int j1, bool second) {
                const double4 p0 = a.posm[j0], p1 = a.posm[j1];
                pair(near, j0, p0);
                if (second) pair(near, j1, p1);
            });
        } else {
            for (int k = sub; k < n; k += G) pair(near, row[k], a.posm[row[k]]);
        }
    };
    if (__all(a.row_r2[i] < B.box.narrow2)) scan(std::true_type{});
    else scan(std::false_type{});
    if constexpr (G > 1) group_sums<G, MFV>(S, pv);
    return density_step(a, i, sub == 0, S, pv, s);
}

// Sweep IT (0 or 1) over the rows, one launch each: nearly every particle of a
// run needs two.  The few that need more leave after the second, so that they
// do not hold a wavefront of finished ones.  IT is a compile-time constant
// because it decides most of the step's branches; both sweeps in one kernel
// spilled 119 registers (2.88 ms for the two at 2.1 M particles).  Three waves
// per SIMD: four spill 28 to 42 registers (0.73 and 0.78 against 0.66 ms).
template <bool MFV, int G, int IT>
__global__ __launch_bounds__(kBlock, 3) void density_stage_kernel(DensityStageArgs a)
{
    const int gt = xcd_block() * kBlock + (int)threadIdx.x;
    const int t = gt / G, sub = gt % G;
    const bool valid = t < a.n_active;
    __shared__ __align__(16) int lds[G == 1 ? kListChunk * kBlock : 1];
    int *chunk = wave_chunk(lds);
    unsigned long long cnt = 0, sweeps = 0;
    int max_iter = 0, left = -1;  // the particle, not done after IT = 1
    const bool packed = G == 1 && IT == 1 && !a.walk_list;  // density_more_kernel follows in the grid
    for_box(a.boxes, a.box_of, valid ? a.active[t] : 0, valid, [&](const BoxDesc &B) {
        const int i = a.active[t];
        const double4 pi = a.posm[i];
        if (!(pi.w > 0)) return;
        if (IT == 1 && a.iter[i] != 1) {  // done, or without a usable row
            if (a.iter[i] == 0) left = i;
            return;
        }
        Iterate s = {a.hsml[i], IT ? a.left[i] : 0.0, IT ? a.right[i] : 0.0, a.cn[i], IT};
        const int n = a.row_n[i];
        const double Rc2 = n <= kDensityCacheCap ? a.row_r2[i] : -1.0;
        bool again = true;
        if (s.h * s.h <= Rc2) {
            again = row_sweep<MFV, G>(a, B, i, pi, n, sub, chunk, s, cnt);
            if (sub == 0) sweeps++;
        }
        if (sub == 0) {
            max_iter = s.iter;
            if (!again) a.iter[i] = kDone;
            else if (IT == 0 && s.iter == 1) hand_on(a, i, s, nullptr, nullptr);
            else if (s.h * s.h <= Rc2 && a.tree.nodes) hand_on(a, i, s, nullptr, nullptr);
            else hand_on(a, i, s, a.walk_list, a.n_walk);
            if (again) left = i;
        }
    });
    if (packed) {
        // up to a quarter of the wavefront goes to the tail list; more wait for density_more_kernel
        const uint64_t bits = __ballot(left >= 0);
        const int n = __popcll(bits), lane = (int)threadIdx.x & 63;
        if (n > 16) {
            if (lane == 0) *a.n_walk = 1;
        } else if (n > 0) {
            int base = 0;
            if (lane == 0) base = atomicAdd(a.n_tail, n);
            base = __shfl(base, 0, 64);
            if (left >= 0) {
                a.tail_list[base + __popcll(bits & ((1ull << lane) - 1))] = left;
                a.iter[left] |= kListed;
            }
        }
    }
    count_sweeps(a, cnt, sweeps, max_iter);
}

// Grid: one sweep of a particle over a walk of its own, G lanes; 1: sweep again, 0:
// done, -1: past the candidate budget (no limit to 64 lanes), the particle as it was.
template <bool MFV, int G>
__device__ __forceinline__ int walk_sweep(const DensityStageArgs &a, const BoxDesc &B, int i, const double4 &pi, int sub,
                                          Iterate &s, unsigned long long &cnt)
{
    const double4 vi = a.velu[i];
    const double h2 = s.h * s.h;
    double hinv, hinv3, hinv4;
    kernel_hinv(s.h, hinv, hinv3, hinv4);
    DensitySums S = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double pv[3] = {0, 0, 0};
    const double xs[3] = {pi.x, pi.y, pi.z};
    unsigned c = 0;
    const bool ok = group_candidates<G>(B, xs, s.h, sub, G < 64 ? a.budget : 0, [&](int j) {
        const double4 pj = a.posm[j];
        double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
        wrap_dp(B.box, dp);
        const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
        if (!(r2 < h2 && pj.w > 0)) return;
        c++;
        density_add<MFV>(dp, r2, pj.w, vi, a.velu[j], hinv, hinv3, hinv4, S, pv);
    });
    if (!ok) return -1;
    cnt += c;
    if constexpr (G > 1) group_sums<G, MFV>(S, pv);
    return density_step(a, i, sub == 0, S, pv, s) ? 1 : 0;
}

// Further sweeps over the rows.  Sets of strongly varying density, and all sets in
// the first stage of a run, where hsml is a guess, leave many particles after two
// (of 250 k in Plummer spheres 196 k need 2.6 more on average, up to 10).  A
// workgroup takes a stretch of the active particles and packs those not converged
// anew for every sweep, so that its wavefronts stay full and keep neighbouring
// particles together; the last few (in the grid the last quarter, and the second sweep's
// wavefronts with as few left list them themselves: a random state of 61^3 has 14 % left,
// density 0.54 ms, with a sixteenth 0.60) go to the tail list.  The 250 k: 0.50 ms
// (stretches of 256 or 1024: 0.67), against 2.0 ms with 16 lanes each to convergence
// and 3.3 ms in four launches over lists whose order the atomics left.
// Tree: a particle whose hsml leaves its row goes to the walk list.  Grid (GRID):
// its row is built anew around the hsml reached, and where that is past the cap (a
// guess far above) or the memory holds no rows, the sweep walks; a walk past the
// candidate budget is done by a wavefront.  Where already the walk for a row passed the
// budget (cells far wider than hsml, in clumps) or has many cells to pass (far smaller
// ones, between clumps) the tail list takes the particle: such walks come thousands to a
// stretch and have to spread over the chip.  With the 16 lanes of the tail walking for
// them, sweep by sweep, the density stage of a 128^3 lattice whose hsml starts 20 %
// low took 35.3 ms, 50 % high 89.6; now 6.7 and 38.0 (a launch per sweep with a lane
// each and no rows: 7.8 and 39.1).  A well guessed 128^3 blast pays under 8 us of 10.7 ms.
// (Stretches of 1024: 61^3 20 % low 1.1 against 0.6 ms.)
template <bool MFV, int G, bool GRID>
__global__ __launch_bounds__(kBlock, 2) void density_more_kernel(DensityStageArgs a)
{
    constexpr int kStretch = 2 * kBlock / G, kFew = kStretch / (GRID ? 4 : 16);
    constexpr int kLists = GRID ? 3 : 2;  // live ones of this sweep and the next, walks past the budget
    if (GRID && *a.n_walk == 0) return;
    __shared__ __align__(16) int lds[GRID ? kRowLds<G> : (G == 1 ? kListChunk * kBlock : 1)];
    __shared__ int live[kLists][kStretch];
    __shared__ int n_live[kLists];
    int *chunk = wave_chunk(lds);
    const int tid = (int)threadIdx.x, lane = tid & 63, sub = tid % G;
    const int first = xcd_block() * kStretch;
    unsigned long long cnt = 0, sweeps = 0;
    int max_iter = 0;
    // keeps i (one lane per entry calls) in list `to`
    auto keep = [&](int to, int i, bool in) {
        const uint64_t bits = __ballot(in);
        int base = 0;
        if (lane == 0 && bits) base = atomicAdd(&n_live[to], __popcll(bits));
        base = __shfl(base, 0, 64);
        if (in) live[to][base + __popcll(bits & ((1ull << lane) - 1))] = i;
    };
    if (tid == 0) n_live[0] = 0;
    __syncthreads();
    for (int k = tid; k < kStretch; k += kBlock) {
        const int t = first + k;
        const int i = t < a.n_active ? a.active[t] : 0;
        // (a particle without mass has no iter)
        bool in = t < a.n_active && (GRID ? (a.iter[i] & (1u << 31 | kListed)) == 0 : a.iter[i] > 0) && a.posm[i].w > 0;
        if (!GRID && in) {
            const double h = a.hsml[i];
            in = a.row_n[i] <= kDensityCacheCap && h * h <= a.row_r2[i];
        }
        keep(0, i, in);
    }
    for (int cur = 0;; cur ^= 1) {
        __syncthreads();
        const int n = n_live[cur];
        if (tid == 0) {
            n_live[cur ^ 1] = 0;
            if (GRID) n_live[kLists - 1] = 0;
        }
        __syncthreads();
        if (n <= kFew) {
            for (int k = tid; k < n; k += kBlock) a.tail_list[atomicAdd(a.n_tail, 1)] = live[cur][k];
            break;
        }
        for (int k0 = 0; k0 < n; k0 += kBlock / G) {
            const int k = k0 + tid / G;
            const bool valid = k < n;
            const int i = valid ? live[cur][k] : 0;
            bool stays = false, wide = false;
            for_box(a.boxes, a.box_of, i, valid, [&](const BoxDesc &B) {
                Iterate s = take_up(a, i);
                const double4 pi = a.posm[i];
                int n_row = a.row_idx ? a.row_n[i] : kNoRow, again = -1;
                if (GRID) {
                    const bool wanted = a.row_idx && row_wanted(n_row, a.row_r2[i], s.h);
                    if ((wanted || n_row > kDensityCacheCap) && many_cells(B.grid, s.h)) n_row = kWideRow;
                    else if (wanted) n_row = grid_row<G>(a, B, i, pi, s.h, sub, lds, 1);
                }
                if (!GRID || n_row <= kDensityCacheCap)
                    again = row_sweep<MFV, G>(a, B, i, pi, n_row, sub, chunk, s, cnt);
                else if (n_row != kWideRow)
                    again = walk_sweep<MFV, G>(a, B, i, pi, sub, s, cnt);
                if (sub != 0) return;
                if (again < 0) {
                    wide = n_row != kWideRow;
                    if (!wide) a.tail_list[atomicAdd(a.n_tail, 1)] = i;
                    return;
                }
                sweeps++;
                max_iter = s.iter > max_iter ? s.iter : max_iter;
                stays = again == 1 && (GRID || s.h * s.h <= a.row_r2[i]);
                if (stays) hand_on(a, i, s, nullptr, nullptr);
                else if (again == 1) hand_on(a, i, s, a.walk_list, a.n_walk);
            });
            keep(cur ^ 1, i, stays);
            if (GRID) keep(kLists - 1, i, wide);
        }
        if constexpr (GRID) {
            __syncthreads();
            const int n_wide = n_live[kLists - 1];
            for (int k = tid / 64; k < n_wide; k += kBlock / 64) {
                const int i = live[kLists - 1][k];
                Iterate s = take_up(a, i);
                const bool stays = walk_sweep<MFV, 64>(a, a.boxes[a.box_of[i]], i, a.posm[i], lane, s, cnt) == 1;
                if (lane == 0) {
                    sweeps++;
                    max_iter = s.iter > max_iter ? s.iter : max_iter;
                    if (stays) {
                        hand_on(a, i, s, nullptr, nullptr);
                        live[cur ^ 1][atomicAdd(&n_live[cur ^ 1], 1)] = i;
                    }
                }
            }
        }
    }
    count_sweeps(a, cnt, sweeps, max_iter);
}

// The listed particles, W lanes each, iterating to convergence: over the
// particle's row while hsml stays inside it (grid: a row built anew once it leaves
// it), else over a walk shared by the lanes.  A walk past the candidate budget (BUDGET)
// leaves the particle to the far list, and any walk (kRowsOnly) to the walk list.  A
// fixed grid strides over the device-side count.
enum DensityWalk { kGridWalk, kTreeWalk, kRowsOnly };
template <bool MFV, int W, bool BUDGET, DensityWalk WALK, int WAVES = 1>
__device__ __forceinline__ void density_iterate(const DensityStageArgs &a, const int *list, const int *count,
                                                WaveWalkLds *walk, int *row_lds = nullptr,
                                                BlockWalkLds<WAVES> *block_walk = nullptr)
{
    const int sub = (int)threadIdx.x % W, part = WAVES > 1 ? (int)threadIdx.x / 64 : 0;
    const int n_groups = WAVES > 1 ? (int)gridDim.x : (int)(gridDim.x * (kBlock / W));
    const int n = *count;
    unsigned long long cnt = 0, sweeps = 0;
    int max_iter = 0;
    for (int u = WAVES > 1 ? (int)blockIdx.x : (int)(blockIdx.x * kBlock + threadIdx.x) / W; u < n; u += n_groups) {
        const int i = list[u];
        const BoxDesc &B = a.boxes[a.box_of[i]];
        const double4 pi = a.posm[i];
        const double4 vi = a.velu[i];
        Iterate s = take_up(a, i);
        int n_row = a.row_n ? a.row_n[i] : kNoRow;
        double tried = a.row_n ? a.row_r2[i] : 0.0, Rc2 = n_row <= kDensityCacheCap ? tried : -1.0;
        const double xs[3] = {pi.x, pi.y, pi.z};
        bool again = true, far = false;
        while (again) {
            const double h2 = s.h * s.h;
            if (WALK == kGridWalk && a.row_n && row_wanted(n_row, tried, s.h)) {
                n_row = grid_row<W>(a, B, i, pi, s.h, sub, row_lds);
                wave_lds_fence();  // the other lanes' entries
                tried = grid_row_r2(s.h);
                Rc2 = n_row <= kDensityCacheCap ? tried : -1.0;
            }
            double hinv, hinv3, hinv4;
            kernel_hinv(s.h, hinv, hinv3, hinv4);
            DensitySums S = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            double pv[3] = {0, 0, 0};
            unsigned long long c = 0;
            auto add = [&](const double4 &pj, const double4 &vj) {
                double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
                wrap_dp(B.box, dp);
                const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                if (!(r2 < h2 && pj.w > 0)) return;
                c++;
                density_add<MFV>(dp, r2, pj.w, vi, vj, hinv, hinv3, hinv4, S, pv);
            };
            if (h2 <= Rc2) {
                const int *row = a.row_idx + (size_t)i * kDensityCacheCap;
                for (int k = sub + W * part; k < n_row; k += W * WAVES) add(a.posm[row[k]], a.velu[row[k]]);
            } else if constexpr (WALK == kRowsOnly) {
                far = true;
                break;
            } else if constexpr (WALK == kTreeWalk) {
                // the loads of one step are used in the next
                double4 pj = make_double4(0, 0, 0, 0), vj = pj;
                auto step = [&](int j, bool valid) {
                    add(pj, vj);
                    pj.w = 0;
                    if (valid) {
                        pj = a.posm[j];
                        vj = a.velu[j];
                    }
                };
                if constexpr (WAVES > 1)
                    block_tree_walk<WAVES>(a.tree, B, xs, s.h, *block_walk, step);
                else
                    far = !wave_tree_walk<false>(a.tree, B, xs, s.h, -1.0, sub, walk[threadIdx.x / 64], step,
                                                 BUDGET ? a.budget : 0);
                if (far) break;
                add(pj, vj);
            } else {
                const int budget = BUDGET ? a.budget : 0;
                if (!group_candidates<W>(B, xs, s.h, sub, budget, [&](int j) { add(a.posm[j], a.velu[j]); })) {
                    far = true;
                    break;
                }
            }
            group_sums<W, MFV>(S, pv);
            if constexpr (WAVES > 1) block_sums<WAVES, MFV>(S, pv);
            cnt += c;
            if (sub == 0 && part == 0) sweeps++;
            again = density_step(a, i, sub == 0 && part == 0, S, pv, s);
        }
        if (sub == 0 && part == 0) {
            if (far && WALK == kRowsOnly) hand_on(a, i, s, a.walk_list, a.n_walk);
            else if (far) hand_on(a, i, s, a.far_list, a.n_far);
            max_iter = s.iter > max_iter ? s.iter : max_iter;
        }
    }
    count_sweeps(a, cnt, sweeps, max_iter);
}

template <bool MFV>
__global__ __launch_bounds__(kBlock, 2) void density_tail_kernel(DensityStageArgs a)
{
    __shared__ int row_lds[kRowLds<kTailLanes>];
    density_iterate<MFV, kTailLanes, true, kGridWalk>(a, a.tail_list, a.n_tail, nullptr, row_lds);
}

template <bool MFV>
__global__ __launch_bounds__(kBlock, 2) void density_far_kernel(DensityStageArgs a)
{
    __shared__ int row_lds[kRowLds<64>];
    density_iterate<MFV, 64, false, kGridWalk>(a, a.far_list, a.n_far, nullptr, row_lds);
}

// Tree: what is left of the rows' sweeps, then the particles that have to walk, a
// wavefront each, and a workgroup for those whose walk passes the candidate budget
// (some hundred of 250 k particles in Plummer spheres, up to 50,000 slots in their
// sweeps).  Those 250 k: walk 0.31 ms, far 0.59 ms (8 wavefronts 0.70), against 3.8
// ms with a wavefront going from node to node.
template <bool MFV>
__global__ __launch_bounds__(kBlock) void density_tree_tail_kernel(DensityStageArgs a)
{
    density_iterate<MFV, kTailLanes, false, kRowsOnly>(a, a.tail_list, a.n_tail, nullptr);
}

template <bool MFV>
__global__ __launch_bounds__(kBlock) void density_tree_walk_kernel(DensityStageArgs a)
{
    __shared__ WaveWalkLds walk[kBlock / 64];
    density_iterate<MFV, 64, true, kTreeWalk>(a, a.walk_list, a.n_walk, walk);
}

template <bool MFV>
__global__ __launch_bounds__(64 * kFarWaves) void density_tree_far_kernel(DensityStageArgs a)
{
    __shared__ BlockWalkLds<kFarWaves> walk;
    density_iterate<MFV, 64, false, kTreeWalk, kFarWaves>(a, a.far_list, a.n_far, nullptr, nullptr, &walk);
}

// no rows: where every active particle starts; the tree's in the walk list
__global__ void density_list_all_kernel(DensityStageArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n_active) return;
    const int i = a.active[t];
    if (!(a.posm[i].w > 0)) return;  // density_isactive: gas with mass > 0 (density.c:85)
    double h = a.hsml[i];
    if ((h < 0) || !isfinite(h) || (h > 0.99 * a.hp.max_hsml)) h = 0.99 * a.hp.max_hsml;  // density.c:484
    const Iterate s = {h, 0, 0, a.cn[i], 0};
    hand_on(a, i, s, a.walk_list, a.n_walk);
    if (!a.walk_list) *a.n_walk = 1;
}

inline unsigned nblocks(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

void launch_density_rows(hipStream_t s, const DensityStageArgs &a)
{
    if (a.n_active <= 0) return;
    const dim3 block(kBlock);
    if (a.tree.nodes)
        hipLaunchKernelGGL(density_tree_rows_kernel, dim3(nblocks((long long)kRowLanes * a.n_active)), block, 0, s, a);
    else if (a.lanes == 8)
        hipLaunchKernelGGL(density_rows_kernel<8>, dim3(nblocks(8LL * a.n_active)), block, 0, s, a);
    else
        hipLaunchKernelGGL(density_rows_kernel<1>, dim3(nblocks(a.n_active)), block, 0, s, a);
}

template <int G, int IT>
static void launch_stage_sweep(hipStream_t s, const DensityStageArgs &a)
{
    const dim3 grid(nblocks((long long)G * a.n_active)), block(kBlock);
    if (a.pvel) hipLaunchKernelGGL((density_stage_kernel<true, G, IT>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((density_stage_kernel<false, G, IT>), grid, block, 0, s, a);
}

void launch_density_stage(hipStream_t s, const DensityStageArgs &a)
{
    if (a.n_active <= 0) return;
    if (!a.row_idx) {
        hipLaunchKernelGGL(density_list_all_kernel, dim3(nblocks(a.n_active)), dim3(kBlock), 0, s, a);
    } else if (a.lanes == 8) {
        launch_stage_sweep<8, 0>(s, a);
        launch_stage_sweep<8, 1>(s, a);
    } else {
        launch_stage_sweep<1, 0>(s, a);
        launch_stage_sweep<1, 1>(s, a);
    }
}

// the counts are on the device: grids that fill the chip, at most one group per particle
template <bool MFV>
static void launch_tree_tail(hipStream_t s, const DensityStageArgs &a)
{
    const dim3 block(kBlock);
    if (a.row_idx) {
        const dim3 grid(nblocks((long long)a.lanes * a.n_active / 2 + a.lanes));
        if (a.lanes == 8) hipLaunchKernelGGL((density_more_kernel<MFV, 8, false>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((density_more_kernel<MFV, 1, false>), grid, block, 0, s, a);
        hipLaunchKernelGGL(density_tree_tail_kernel<MFV>, dim3(std::min(2048u, nblocks((long long)kTailLanes * a.n_active))),
                           block, 0, s, a);
    }
    hipLaunchKernelGGL(density_tree_walk_kernel<MFV>, dim3(std::min(2048u, nblocks(64LL * a.n_active))), block, 0, s, a);
    if (a.budget)
        hipLaunchKernelGGL(density_tree_far_kernel<MFV>, dim3(std::min(512, a.n_active)), dim3(64 * kFarWaves), 0, s, a);
}

template <bool MFV>
static void launch_grid_tail(hipStream_t s, const DensityStageArgs &a)
{
    // the counts are on the device: enough workgroups to fill the chip, at most one group per particle
    const dim3 block(kBlock), waves(std::min(2048u, nblocks(64LL * a.n_active)));
    if (a.lanes == 8) {
        // few particles: the whole tail with a wavefront each, in one launch (a nearly
        // empty tail of 32 k particles: 5.1 us against 4.1 + 3.5 and the gap between)
        DensityStageArgs b = a;
        b.far_list = a.tail_list;
        b.n_far = a.n_tail;
        hipLaunchKernelGGL(density_far_kernel<MFV>, waves, block, 0, s, b);
        return;
    }
    if (!a.walk_list)
        hipLaunchKernelGGL((density_more_kernel<MFV, 1, true>), dim3(nblocks((long long)a.n_active / 2 + 1)), block, 0, s, a);
    hipLaunchKernelGGL(density_tail_kernel<MFV>, dim3(std::min(2048u, nblocks((long long)kTailLanes * a.n_active))), block, 0,
                       s, a);
    if (a.budget) hipLaunchKernelGGL(density_far_kernel<MFV>, waves, block, 0, s, a);
}

void launch_density_tail(hipStream_t s, const DensityStageArgs &a)
{
    if (a.n_active <= 0) return;
    if (a.tree.nodes) {
        if (a.pvel) launch_tree_tail<true>(s, a);
        else launch_tree_tail<false>(s, a);
        return;
    }
    if (a.pvel) launch_grid_tail<true>(s, a);
    else launch_grid_tail<false>(s, a);
}

}  // namespace gzm
