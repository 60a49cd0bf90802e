// gzm_kernels.hip -- HIP kernels of the MFM hydro pass for gfx950 (FP64).
//
// "Gather form": one lane or a small group of lanes per active particle i
// evaluates every pair (i, j) for its own particle only -- from the candidate
// rows of the density stage (gzm_density.hip) or the pair list where they hold
// the set, else over a walk of the grid or tree -- and finishes the particle's
// work (gradient construction + limiter, flux sums -> dv/dt, du/dt).
// Consecutive lanes hold consecutive particles of the Morton-sorted order, so
// those of a wavefront meet almost the same neighbours and their loads hit the
// same cache lines.
//
// No pair writes to j (the reference disables its pair-symmetric writes too,
// hydro_evaluate.h:159-168, gradients.c:1554-1565), so every kernel is free of
// races and deterministic for a fixed particle order.
#include "grid_device.h"
#include "gzm_internal.h"

namespace gzm {

namespace {

// ---------------------------------------------------------------------------
// grid build
// ---------------------------------------------------------------------------
// global cell index of a position in box B (cell_base + linear cell id)
__device__ __forceinline__ int global_cell(const BoxDesc &B, double x, double y, double z)
{
    const Grid &g = B.grid;
    return B.cell_base + (cell_coord(x, g.inv_s[0], g.nc[0]) * g.nc[1] + cell_coord(y, g.inv_s[1], g.nc[1])) * g.nc[2] +
           cell_coord(z, g.inv_s[2], g.nc[2]);
}

// sort key: box index above the 30-bit Morton code of the cell in its box
__global__ void cell_keys_kernel(int n, const double *pos, const BoxDesc *boxes, const int *box_caller,
                                 uint64_t *keys, int *iota)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = box_caller ? box_caller[i] : 0;
    const Grid &g = boxes[b].grid;
    int cx = cell_coord(pos[3 * i + 0], g.inv_s[0], g.nc[0]);
    int cy = cell_coord(pos[3 * i + 1], g.inv_s[1], g.nc[1]);
    int cz = cell_coord(pos[3 * i + 2], g.inv_s[2], g.nc[2]);
    keys[i] = ((uint64_t)b << 30) | morton3(cx, cy, cz);
    iota[i] = i;
}

__global__ void gather_sorted_kernel(int n, const int *perm, const double *pos, const double *vel,
                                     const double *mass, const double *u, const BoxDesc *boxes, const int *box_caller,
                                     double4 *posm, double4 *velu, float4 *posf, int *inv, int *box_of)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = perm[k];
    posm[k] = make_double4(pos[3 * i + 0], pos[3 * i + 1], pos[3 * i + 2], mass[i]);
    velu[k] = make_double4(vel[3 * i + 0], vel[3 * i + 1], vel[3 * i + 2], u[i]);
    const int b = box_caller ? box_caller[i] : 0;
    if (posf) {
        const double s = boxes[b].unit;
        posf[k] = make_float4((float)(pos[3 * i + 0] * s), (float)(pos[3 * i + 1] * s), (float)(pos[3 * i + 2] * s),
                              mass[i] > 0 ? 1.0f : 0.0f);
    }
    inv[i] = k;
    box_of[k] = b;
}

__global__ void gather_scalar_kernel(int n, const int *perm, const double *src, double *dst, int width)
{
    long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * width) return;
    int k = (int)(t / width), c = (int)(t % width);
    dst[t] = src[(long long)perm[k] * width + c];
}

// Fields from sorted slots into caller order, all in one launch: consecutive
// threads write consecutive elements, so that the destination may be host memory
// (the writes then cross the bus as they are made, with no copy after them).
__global__ __launch_bounds__(kBlock) void export_kernel(ExportArgs a)
{
    int q = 0;
    while (q + 1 < a.n_fields && blockIdx.x >= a.first_block[q + 1]) q++;
    const ExportField f = a.field[q];
    const long long t = (long long)(blockIdx.x - a.first_block[q]) * kBlock + threadIdx.x;
    if (t >= (long long)a.n * f.w) return;
    const int i = (int)(t / f.w), c = (int)(t % f.w);
    // (row, column) of the full matrix -> 00 01 02 11 12 22
    const int e = f.w == 9 && f.w_src == 6 ? (c == 8 ? 5 : c / 3 + c % 3 + (c == 4 || c == 5 || c == 7 ? 1 : 0)) : c;
    f.dst[t] = f.src[(long long)a.inv[i] * f.w_src + f.off + e];
}

__global__ void export_u8_kernel(int n, const int *inv, const uint8_t *src, uint8_t *dst)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[inv[i]];
}

__global__ void fill_fields_kernel(FillArgs a)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.n) return;
    for (int q = 0; q < a.n_fills; q++)
        for (int c = 0; c < a.width[q]; c++) a.p[q][(size_t)c * a.n + k] = a.value[q];
}

__global__ void iota_kernel(int n, int *p)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = k;
}

__global__ void restore_kernel(int n, double *hsml, const double *hsml0, double *cn, const double *cn0, double *vsig,
                               const double *vsig0, double *dmass, const double *dmass0)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    hsml[k] = hsml0[k];
    cn[k] = cn0[k];
    vsig[k] = vsig0[k];
    if (dmass0) dmass[k] = dmass0[k];
}

// the sum of a stage's kCtrSpread counter copies, one lane each, into host memory
__global__ void publish_counters_kernel(const Counters *ctr, Counters *host)
{
    Counters h = ctr[threadIdx.x];
    for (int off = 32; off > 0; off >>= 1) {
        h.interactions += __shfl_xor(h.interactions, off, 64);
        h.retries += __shfl_xor(h.retries, off, 64);
        h.exact_calls += __shfl_xor(h.exact_calls, off, 64);
        h.updates += __shfl_xor(h.updates, off, 64);
        h.redo_n += __shfl_xor(h.redo_n, off, 64);
        h.overflow_slices += __shfl_xor(h.overflow_slices, off, 64);
        h.deferred += __shfl_xor(h.deferred, off, 64);
        h.status = max(h.status, __shfl_xor(h.status, off, 64));
        h.sweeps = max(h.sweeps, __shfl_xor(h.sweeps, off, 64));
    }
    if (threadIdx.x == 0) *host = h;
}

__global__ void cell_ranges_kernel(int n, const double4 *posm, const BoxDesc *boxes, const int *box_of, int2 *range)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    double4 p = posm[k];
    const int c = global_cell(boxes[box_of[k]], p.x, p.y, p.z);
    int cprev = -1, cnext = -1;
    if (k > 0) {
        double4 q = posm[k - 1];
        cprev = global_cell(boxes[box_of[k - 1]], q.x, q.y, q.z);
    }
    if (k + 1 < n) {
        double4 q = posm[k + 1];
        cnext = global_cell(boxes[box_of[k + 1]], q.x, q.y, q.z);
    }
    if (c != cprev) range[c].x = k;
    if (c != cnext) range[c].y = k + 1;
}

__global__ void clear_box_hmax_kernel(int n_boxes, BoxDesc *boxes, Counters *ctr)
{
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < n_boxes) boxes[b].hmax = 0.0;
    if (ctr && b < kCtrSpread) ctr[b] = Counters{};
}

__global__ void flag_unconverged_kernel(const int *n_live_dev, Counters *ctr)
{
    if (threadIdx.x == 0 && *n_live_dev > 0) atomicMax(&ctr->status, 1155);
}

__global__ void clear_counters_kernel(Counters *ctr)
{
    ctr[threadIdx.x] = Counters{};  // kCtrSpread threads
}

__global__ void density_begin_kernel(Counters *ctr, int *counts)
{
    if (threadIdx.x >= 1 && threadIdx.x < kDensityCounts) counts[threadIdx.x] = 0;
    if (ctr) ctr[threadIdx.x] = Counters{};  // kCtrSpread threads
}

__global__ void map_active_kernel(int n_active, const int *active_caller, const int *inv, int *active_sorted)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_active) return;
    active_sorted[t] = inv[active_caller[t]];
}

__global__ void fill_int_kernel(int *p, int n, int v)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

__global__ void fill_u8_kernel(uint8_t *p, int n, uint8_t v)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

__global__ void set_flags_kernel(int n_active, const int *active, uint8_t *flags)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n_active) flags[active[t]] = 1;
}

// ---------------------------------------------------------------------------
// density (density.c:252-347 pair sums + 505-850 iteration, fused): the parts
// that the FP32 sweeps of precision 2 use; precisions 0 and 1 have gzm_density.hip
// ---------------------------------------------------------------------------
__global__ void density_init_kernel(int n_active, const int *active, const double4 *posm, double *hsml, double *left,
                                    double *right, double max_hsml, int *live_flag)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_active) return;
    int i = active[t];
    int live = posm[i].w > 0;  // density_isactive: gas with mass > 0 (density.c:85)
    live_flag[t] = live;
    if (!live) return;
    left[i] = 0;
    right[i] = 0;
    double h = hsml[i];
    if ((h < 0) || !isfinite(h) || (h > 0.99 * max_hsml)) hsml[i] = 0.99 * max_hsml;  // density.c:484
}

// one density pair (density.c:252-347): j's terms into S when r_ij < h_i.
// Also sets `edge` when r_ij^2 lies within kEdgeBand of h_i^2.
__device__ __forceinline__ bool density_pair(const BoxDesc &G, const double4 &pi, const double4 &vi,
                                             const DensitySweepArgs &a, int j, double h2, double hinv,
                                             double hinv3, double hinv4, DensitySums &S, bool &edge)
{
    const double4 pj = a.posm[j];
    double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
    wrap_dp(G.box, dp);
    const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
    if (pj.w > 0 && fabs(r2 - h2) <= kEdgeBand * h2) edge = true;
    if (!(r2 < h2 && pj.w > 0)) return false;
    const double r = sqrt(r2);
    const double u = r * hinv;
    double wk, dwk;
    kernel_wdw(u, hinv3, hinv4, wk, dwk);
    S.ngb += wk;
    S.rho += pj.w * wk;
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
        const double4 vj = a.velu[j];
        const double dv0 = vi.x - vj.x, dv1 = vi.y - vj.y, dv2 = vi.z - vj.z;
        S.divvel -= dwk * (dp[0] * dv0 + dp[1] * dv1 + dp[2] * dv2) / r;
    }
    return true;
}

// the hsml update of one particle from its sums, and its outputs; returns
// hsml_update's result (1 sweep again, 0 done, -1 bracket failure)
__device__ __forceinline__ int density_store(const DensitySweepArgs &a, int t, int i, double h, const DensitySums &S)
{
    double left = a.left[i], right = a.right[i];
    DensityResult R;
    const int res = hsml_update(a.hp, S, h, left, right, a.cn[i], R);
    a.hsml[i] = h;
    a.left[i] = left;
    a.right[i] = right;
    a.cn[i] = R.cn_stored;
    a.num_ngb[i] = R.num_ngb;
    a.dhsml[i] = R.dhsml;
    a.divvel[i] = R.divvel;
    a.rho[i] = R.rho_sum;
    a.fce[i] = R.fce;
#pragma unroll
    for (int k = 0; k < 6; k++) a.nvt[6 * (size_t)i + k] = R.nvt[k];
    a.redo[t] = (res == 1) ? 1 : 0;
    if (res < 0) atomicMax(&ctr_slot(a.ctr)->status, (int)6);
    return res;
}

// The particles that passed the candidate budget: one wavefront each, its
// lanes sharing the walk (wave_candidates); the sums are reduced across the
// wavefront (another summation order than a single lane's, FP64 throughout).
// A fixed grid strides over the list, so the launch is sized independently of
// the (device-side) count.
__global__ __launch_bounds__(kBlock) void density_heavy_kernel(DensitySweepArgs a)
{
    __shared__ WaveWalkLds walk[kBlock / 64];
    const int lane = threadIdx.x & 63;
    const int n_waves = (int)(gridDim.x * (kBlock / 64));
    const int n = a.wave_all ? (a.n_live_dev ? *a.n_live_dev : a.n_live) : *a.n_heavy;
    if (a.wave_all && a.n_live_dev) {  // captured pass: clear the flags up to the capacity
        for (int t = n + (int)(blockIdx.x * kBlock + threadIdx.x); t < a.n_live; t += (int)(gridDim.x * kBlock))
            a.redo[t] = 0;
    }
    for (int u = (int)((blockIdx.x * kBlock + threadIdx.x) >> 6); u < n; u += n_waves) {
        const int t = a.wave_all ? u : a.heavy_list[u];
        const int i = a.live[t];
        const BoxDesc &G = a.boxes[a.box_of[i]];
        const double4 pi = a.posm[i];
        const double4 vi = a.velu[i];
        const double h = a.hsml[i];
        double hinv, hinv3, hinv4;
        kernel_hinv(h, hinv, hinv3, hinv4);
        const double h2 = h * h;
        DensitySums S = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        const double xs[3] = {pi.x, pi.y, pi.z};
        unsigned long long c = 0;
        bool edge = false;
        wave_candidates(a.tree, G, xs, h, lane, walk[threadIdx.x >> 6], [&](int j) {
            if (density_pair(G, pi, vi, a, j, h2, hinv, hinv3, hinv4, S, edge)) c++;
        });
        const bool any_edge = __any(edge);
        S.ngb = wave_sum(S.ngb); S.rho = wave_sum(S.rho); S.dhsml = wave_sum(S.dhsml);
        S.divvel = wave_sum(S.divvel);
        S.t00 = wave_sum(S.t00); S.t01 = wave_sum(S.t01); S.t02 = wave_sum(S.t02);
        S.t11 = wave_sum(S.t11); S.t12 = wave_sum(S.t12); S.t22 = wave_sum(S.t22);
        S.f0 = wave_sum(S.f0); S.f1 = wave_sum(S.f1); S.f2 = wave_sum(S.f2);
        wave_add_u64(&ctr_slot(a.ctr)->interactions, c);
        if (lane == 0) {
            const int res = density_store(a, t, i, h, S);
            if (res == 0 && any_edge) a.edge_list[atomicAdd(a.n_edge, 1)] = i;
        }
    }
}

__global__ void edge_reset_kernel(int cap, const int *n_edge, const int *edge_list, const double *hsml_entry,
                                  double *hsml, double *left, double *right, int *iter)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cap || t >= *n_edge) return;
    const int i = edge_list[t];
    hsml[i] = hsml_entry[i];
    left[i] = 0;
    right[i] = 0;
    iter[i] = 0;
}

__global__ void density_finalize_kernel(int n_active, const int *active, const double4 *posm, const double4 *velu,
                                        const double *hsml, double *num_ngb, double *rho, double *pres, double gm1)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_active) return;
    int i = active[t];
    double m = posm[i].w;
    if (!(m > 0)) return;
    double h = hsml[i], nn = num_ngb[i], d;
    // density.c:967-978 (MFM: own mass times the kernel number density)
    if ((h > 0) && (nn > 0)) d = m * nn / (kNormCoeff * cube(h));
    else if (h <= 0) d = 0;
    else d = m / (kNormCoeff * cube(h));
    rho[i] = d;
    pres[i] = gm1 * velu[i].w * d;  // eos.c:58-61
    num_ngb[i] = (nn > 0) ? cbrt(nn) : 0;  // density.c:1020
}

// ---------------------------------------------------------------------------
// gradients (gradients.c:1477-2089 pair loop, 1052-1253 finalize)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void pack_grad(int k, const double4 *posm, const double4 *velu, const double *hsml,
                                          const double *rho, const double *pres, double4 *xh, GradRec *rec)
{
    double4 p = posm[k], v = velu[k];
    GradRec r;
    xh[k] = make_double4(p.x, p.y, p.z, hsml[k]);
    r.vr = make_double4(v.x, v.y, v.z, rho[k]);
    r.pm = make_double2(pres[k], p.w);
    rec[k] = r;
}

// One particle's FP64 force record (shared by pack_force_kernel and the
// gradient kernel's epilogue, so that both write the same bits)
__device__ __forceinline__ ForceRec make_force_rec(const double4 &p, const double4 &v, double d, double P, double h,
                                                   double dh, double cn, double fce, const double *t, const double *g,
                                                   double gamma)
{
    ForceRec r;
    r.v[0] = v.x; r.v[1] = v.y; r.v[2] = v.z;
    r.h = h; r.hinv = 1.0 / h;
    r.rho = d; r.P = P;
    r.cs = sqrt(gamma * P / d);  // eos.c:245-254
    r.V = p.w / d; r.dhsml = dh; r.fce = fce;
    for (int k = 0; k < 6; k++) r.nvt[k] = t[k];
    for (int k = 0; k < 3; k++) { r.gr[k] = g[k]; r.gp[k] = g[3 + k]; }
    for (int k = 0; k < 9; k++) r.gv[k] = g[6 + k];
    r.cn = cn; r.e = P / d;
    return r;
}

// What the pair stages read that hsml decides, in one launch of three parts by
// workgroup: the largest hsml of each box (the search radius of the pair loops,
// force_update_hmax), one tile of up to kHmaxTile slots of a box each (block
// maximum, then one atomic max on the bit pattern, valid for hsml >= 0); that of
// each cell, rounded up; and the FP64 gradient records (a.rec NULL: none).
__global__ __launch_bounds__(kBlock) void pair_prepare_kernel(PairPrepareArgs a)
{
    __shared__ double red[kBlock / 64];
    int block = blockIdx.x;
    if (block < a.n_tiles) {
        const int2 tile = a.tiles[block];  // (box, first slot)
        const BoxDesc &B = a.boxes[tile.x];
        const int end = min(tile.y + kHmaxTile, B.first + B.count);
        double m = 0;
        for (int k = tile.y + threadIdx.x; k < end; k += kBlock) m = fmax(m, a.hsml[k]);
        for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < kBlock / 64; w++) m = fmax(m, red[w]);
            atomicMax((unsigned long long *)&a.boxes[tile.x].hmax, (unsigned long long)__double_as_longlong(m));
        }
        return;
    }
    block -= a.n_tiles;
    if (block < a.cell_blocks) {
        const int c = block * kBlock + (int)threadIdx.x;
        if (c >= a.n_cells) return;
        const int2 r = a.range[c];
        double m = 0.0;
        for (int k = r.x; k < r.y; ++k) m = (a.hsml[k] > m) ? a.hsml[k] : m;
        a.cell_hmax[c] = __double2float_ru(m);
        return;
    }
    const int k = (block - a.cell_blocks) * kBlock + (int)threadIdx.x;
    if (k < a.n) pack_grad(k, a.posm, a.velu, a.hsml, a.rho, a.pres, a.xh, a.rec);
}

constexpr int kNoSlot = 0x7fffffff;  // above every sorted slot: the end of a merged row

// Symmetric pair rows: particle j offers itself to particle i (0 < r_ij < h_j)
// unless j is in i's candidate row (r_ij below the row's radius) or i's row
// does not cover its own hsml (then i walks the tree anyway).
__device__ __forceinline__ void sym_offer(const SymRowArgs &a, const BoxDesc &G, const double4 &pj, double hj2, int j,
                                          int i)
{
    const double4 pi = a.posm[i];
    // r_ij as the gradient kernel computes it for i (x_i - x_j)
    double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
    wrap_dp(G.box, dp);
    const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
    if (!(r2 < hj2) || r2 <= 0) return;
    const double ri2 = a.dcache_r2[i];
    if (r2 < ri2) return;
    if (a.dcache_n[i] > kDensityCacheCap) return;
    const double h_i = a.hsml[i];
    if (!(h_i * h_i <= ri2)) return;
    const int k = atomicAdd(&a.bcount[i], 1);
    if (k < kPairRowCap) a.brow[(size_t)i * kPairRowCap + k] = j;
}

// Symmetric pair rows, scatter: each j takes the i from its own candidate row
// when that covers h_j; the other j (rows past their cap, hsml past the row's
// radius) are listed for sym_rows_wave_kernel.
__global__ __launch_bounds__(kBlock) void sym_rows_scatter_kernel(SymRowArgs a)
{
    const int j = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = j < a.n;
    for_box(a.boxes, a.box_of, valid ? j : 0, valid, [&](const BoxDesc &G) {
        const double4 pj = a.posm[j];
        const double h_j = a.hsml[j];
        if (!(h_j > 0)) return;
        const double hj2 = h_j * h_j;
        const int n_j = a.dcache_n[j];
        if (n_j <= kDensityCacheCap && hj2 <= a.dcache_r2[j]) {
            const int *row = a.dcache_idx + (size_t)j * kDensityCacheCap;
            for (int k = 0; k < n_j; k++) sym_offer(a, G, pj, hj2, j, row[k]);
        } else {
            a.wlist[atomicAdd(a.wcount, 1)] = j;
        }
    });
}

// The listed j, one wavefront each: its lanes share the tree walk of radius h_j
// (wave_candidates).  A fixed grid strides over the device-side count.
__global__ __launch_bounds__(kBlock) void sym_rows_wave_kernel(SymRowArgs a)
{
    __shared__ WaveWalkLds walk[kBlock / 64];
    const int lane = threadIdx.x & 63;
    const int n_waves = (int)(gridDim.x * (kBlock / 64));
    const int n = *a.wcount;
    for (int u = (int)((blockIdx.x * kBlock + threadIdx.x) >> 6); u < n; u += n_waves) {
        const int j = a.wlist[u];
        const BoxDesc &G = a.boxes[a.box_of[j]];
        const double4 pj = a.posm[j];
        const double h_j = a.hsml[j];
        const double hj2 = h_j * h_j;
        const double xs[3] = {pj.x, pj.y, pj.z};
        wave_candidates(a.tree, G, xs, h_j, lane, walk[threadIdx.x >> 6], [&](int i) { sym_offer(a, G, pj, hj2, j, i); });
    }
}

// Symmetric pair rows, sort: each row ascending (a handful of entries)
__global__ __launch_bounds__(kBlock) void sym_rows_sort_kernel(int n, int *brow, const int *bcount)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int c = bcount[i];
    if (c < 2 || c > kPairRowCap) return;
    int *r = brow + (size_t)i * kPairRowCap;
    for (int k = 1; k < c; k++) {
        const int v = r[k];
        int m = k - 1;
        while (m >= 0 && r[m] > v) {
            r[m + 1] = r[m];
            m--;
        }
        r[m + 1] = v;
    }
}

// where a gradient kernel takes its candidates from: a walk (grid or tree), the
// tree's candidate and pair rows, the grid's candidate rows (the last two fall
// back to the walk for a particle whose rows do not hold its pair set)
enum GradSource { kFromWalk, kFromTreeRows, kFromGridRows };

// One particle's sums of the gradient loop: g as stored (rho, P, v rows), the
// extremes of the differences (rho, P, v), the largest distance.
struct GradSums {
    double g[15], mn[5], mx[5], maxd;
};

// NV_T, the limiter (SELFGRAVITY_OFF, no MAGNETIC/GALSF: h_lim = h, stol = 0.1;
// gradients.c:1219-1232) and, with every particle active, the force record that
// pack_force_kernel would write
__device__ __forceinline__ void finish_gradients(const GradientArgs &a, int i, const double4 &xi, const GradRec &ri,
                                                 GradSums &S, double g_out[15], ForceRec &f_out)
{
    const double h_i = xi.w, rho_i = ri.vr.w, p_i = ri.pm.x, m_i = ri.pm.y;
    double nvt[6];
#pragma unroll
    for (int k = 0; k < 6; k++) nvt[k] = a.nvt[6 * (size_t)i + k];
#pragma unroll
    for (int q = 0; q < 5; q++) apply_nvt(nvt, S.g + 3 * q);
    const double cn = a.cn[i];
    const double d_max = (h_i > S.maxd) ? h_i : S.maxd;
    double a_lim = 0.25;
    if (cn > 100) a_lim = dmin(0.5, 0.25 + 0.25 * (cn - 100) / 100);
    slope_limit(S.g + 0, S.mx[0], S.mn[0], a_lim, h_i, 0, 1, d_max, rho_i);
    slope_limit(S.g + 3, S.mx[1], S.mn[1], a_lim, h_i, 0.1, 1, d_max, p_i);
    slope_limit(S.g + 6, S.mx[2], S.mn[2], a_lim, h_i, 0.1, 0, 0, 0);
    slope_limit(S.g + 9, S.mx[3], S.mn[3], a_lim, h_i, 0.1, 0, 0, 0);
    slope_limit(S.g + 12, S.mx[4], S.mn[4], a_lim, h_i, 0.1, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < 15; k++) g_out[k] = S.g[k];
    if (a.frec_out)
        f_out = make_force_rec(make_double4(xi.x, xi.y, xi.z, m_i), make_double4(ri.vr.x, ri.vr.y, ri.vr.z, 0.0),
                               rho_i, p_i, h_i, a.dhsml[i], cn, a.fce[i], nvt, S.g, a.gamma);
}

// Bound by the L2 reads of the neighbours (5,500 lines per wavefront before the
// split of GradRec and the chunked row reads): of 2.1 M particles 2.36 ms from
// the walk, 1.72 from the rows entry by entry, 1.27 with rows read 64 bytes at
// a time, positions apart from the rest of the record, and whole-record stores.
//
// G lanes per particle (more than one for few particles, which would leave most
// SIMDs without a wavefront): each takes every G-th candidate, the sums are
// reduced at the end and every lane finishes the particle (32^3 particles: 0.036
// against 0.145 ms from the walk with one lane).
template <int BS, GradSource SRC, int G = 1>
__global__ __launch_bounds__(BS, 3) void gradients_kernel(GradientArgs a)
{
    // Pair-list entries are staged in LDS and leave as whole 64-byte chunks:
    // single 4-byte stores spread over the loop would reach HBM as partial-line
    // write-backs.  BS = blockDim.x.  With G > 1 the entries of a step are packed
    // by ballot and adjoin anyway.
    __shared__ __align__(16) int lds[G == 1 ? kListChunk * BS : 1];
    __shared__ __align__(16) int lds_row[G == 1 && SRC == kFromGridRows ? kListChunk * BS : 1];
    int *stage = wave_chunk(lds), *chunk = wave_chunk(lds_row);
    const int t = (xcd_block() * BS + (int)threadIdx.x) / G, sub = (int)threadIdx.x % G;
    bool valid = t < a.n_active;
    unsigned long long cnt = 0;
    int listed = 0, out_i = 0;
    double g_out[15];  // the particle's gradients and force record, stored by the whole wavefront
    ForceRec f_out;
    for_box(a.boxes, a.box_of, valid ? a.active[t] : 0, valid, [&](const BoxDesc &B) {
        const int i = a.active[t];
        out_i = i;
        const GradRec ri = a.rec[i];
        const double4 xi = a.xh[i];
        double gr0 = 0, gr1 = 0, gr2 = 0, gp0 = 0, gp1 = 0, gp2 = 0;
        double gv00 = 0, gv01 = 0, gv02 = 0, gv10 = 0, gv11 = 0, gv12 = 0, gv20 = 0, gv21 = 0, gv22 = 0;
        double maxd = 0, mn_r = 0, mx_r = 0, mn_p = 0, mx_p = 0;
        double mn_v0 = 0, mx_v0 = 0, mn_v1 = 0, mx_v1 = 0, mn_v2 = 0, mx_v2 = 0;
        const double h_i = xi.w, rho_i = ri.vr.w, p_i = ri.pm.x, m_i = ri.pm.y;
        int *list_row = a.list.idx ? a.list.idx + (size_t)t * a.list.cap : nullptr;
        if ((m_i > 0) && (rho_i > 0) && (h_i > 0)) {  // GasGrad_isactive (gradients.c:66-75)
            double hinv, hinv3, hinv4;
            kernel_hinv(h_i, hinv, hinv3, hinv4);
            const double h2_i = h_i * h_i;
            const double xs[3] = {xi.x, xi.y, xi.z};
            // the force loop's pair set (hydro_evaluate.h:149-150)
            auto is_pair = [&](auto near, const double4 &xj, const GradRec &rj, double dp[3], double &r2) {
                dp[0] = xs[0] - xj.x;
                dp[1] = xs[1] - xj.y;
                dp[2] = xs[2] - xj.z;
                if constexpr (near.value) wrap_near(B.box, dp);
                else wrap_dp(B.box, dp);
                r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                if (r2 <= 0) return false;
                if ((r2 >= h2_i) && (r2 >= xj.w * xj.w)) return false;
                return (rj.pm.y > 0) && (rj.vr.w > 0);
            };
            // list entry (m_j > 0, rho_j > 0; gradients also need h_j > 0)
            auto enlist = [&](int j, bool in) {
                if (!list_row) return;
                if constexpr (G == 1) {
                    if (!in) return;
                    if (listed < a.list.cap) {
                        const int c = listed & (kListChunk - 1);
                        stage[c * 64 + (threadIdx.x & 63)] = j;
                        if (c == kListChunk - 1) flush_list_chunk(stage, list_row + (listed - c));
                    }
                    listed++;
                } else {
                    const unsigned bits = (unsigned)(__ballot(in) >> ((threadIdx.x & 63) & ~(G - 1))) & ((1u << G) - 1);
                    const int k = listed + __popc(bits & ((1u << sub) - 1));
                    if (in && k < a.list.cap) list_row[k] = j;
                    listed += __popc(bits);
                }
            };
            auto add = [&](const double4 &xj, const GradRec &rj, const double dp[3], double r2) {
                const double h_j = xj.w;
                const double4 vr = rj.vr;
                const double2 pm = rj.pm;
                if (!(h_j > 0)) return;
                cnt++;
                const double r = sqrt(r2);
                const double wk_i = (r < h_i) ? kernel_w(r * hinv, hinv3) : 0.0;
                if (r > maxd) maxd = r;
                const double d_rho = vr.w - rho_i;
                minmax_check(d_rho, mn_r, mx_r);
                const double dpp = pm.x - p_i;
                minmax_check(dpp, mn_p, mx_p);
                const double dv0 = vr.x - ri.vr.x, dv1 = vr.y - ri.vr.y, dv2 = vr.z - ri.vr.z;
                minmax_check(dv0, mn_v0, mx_v0);
                minmax_check(dv1, mn_v1, mx_v1);
                minmax_check(dv2, mn_v2, mx_v2);
                if (r < h_i) {
                    const double w0 = -wk_i * dp[0], w1 = -wk_i * dp[1], w2 = -wk_i * dp[2];
                    gr0 += w0 * d_rho; gr1 += w1 * d_rho; gr2 += w2 * d_rho;
                    gp0 += w0 * dpp; gp1 += w1 * dpp; gp2 += w2 * dpp;
                    gv00 += w0 * dv0; gv01 += w1 * dv0; gv02 += w2 * dv0;
                    gv10 += w0 * dv1; gv11 += w1 * dv1; gv12 += w2 * dv1;
                    gv20 += w0 * dv2; gv21 += w1 * dv2; gv22 += w2 * dv2;
                }
            };
            auto visit = [&](int j) {
                const double4 xj = a.xh[j];
                double dp[3], r2;
                if (!is_pair(std::false_type{}, xj, a.rec[j], dp, r2)) return;
                enlist(j, true);
                add(xj, a.rec[j], dp, r2);
            };
            // G > 1: candidate k + sub of a run of `end` for each lane, all lanes in step
            auto visit_step = [&](auto near, int j, bool valid_j) {
                double dp[3], r2;
                double4 xj;
                bool in = valid_j;
                if (in) {
                    xj = a.xh[j];
                    in = is_pair(near, xj, a.rec[j], dp, r2);
                }
                enlist(j, in);
                if (in) add(xj, a.rec[j], dp, r2);
            };
            const int n_a = SRC != kFromWalk ? a.dcache_n[i] : kDensityCacheCap + 1;
            const int n_b = SRC == kFromTreeRows ? a.bcount[i] : 0;
            if (SRC == kFromGridRows && n_a <= kDensityCacheCap && row_holds_pairs(B, xs, h_i, a.dcache_r2[i])) {
                const int *row = a.dcache_idx + (size_t)i * kDensityCacheCap;
                auto scan = [&](auto near) {
                    if constexpr (G > 1) {
                        for (int k = 0; k < n_a; k += G) visit_step(near, row[min(k + sub, n_a - 1)], k + sub < n_a);
                    } else {
                        for_row_pairs(chunk, row, n_a, [&](int j0, int j1, bool second) {
                            const double4 x0 = a.xh[j0], x1 = a.xh[j1];
                            double dp[3], r2;
                            if (is_pair(near, x0, a.rec[j0], dp, r2)) {
                                enlist(j0, true);
                                add(x0, a.rec[j0], dp, r2);
                            }
                            if (second && is_pair(near, x1, a.rec[j1], dp, r2)) {
                                enlist(j1, true);
                                add(x1, a.rec[j1], dp, r2);
                            }
                        });
                    }
                };
                if (__all(a.dcache_r2[i] * 1.01 < B.box.narrow2)) scan(std::true_type{});
                else scan(std::false_type{});
            } else if (SRC == kFromTreeRows && n_a <= kDensityCacheCap && h2_i <= a.dcache_r2[i] && n_b <= kPairRowCap) {
                // ascending merge of i's candidate row and its pair row
                const int *ra = a.dcache_idx + (size_t)i * kDensityCacheCap;
                const int *rb = a.brow + (size_t)i * kPairRowCap;
                int ka = 0, kb = 0;
                int ja = (n_a > 0) ? ra[0] : kNoSlot, jb = (n_b > 0) ? rb[0] : kNoSlot;
                while (ka < n_a || kb < n_b) {
                    if (ja < jb) {
                        visit(ja);
                        ka++;
                        ja = (ka < n_a) ? ra[ka] : kNoSlot;
                    } else {
                        visit(jb);
                        kb++;
                        jb = (kb < n_b) ? rb[kb] : kNoSlot;
                    }
                }
            } else if constexpr (SRC == kFromTreeRows) {  // left to gradients_walk_kernel
                a.far_list[atomicAdd(a.n_far, 1)] = t;
                valid = false;
                return;
            } else if constexpr (G > 1) {
                const double R = (B.hmax > h_i) ? B.hmax : h_i;
                bool full[3];
                for_each_cell(B.grid, xs, R, full, [&](int, int, int, int beg, int end) {
                    for (int k = beg; k < end; k += G) visit_step(std::false_type{}, k + sub, k + sub < end);
                }, h_i);
            } else {
                const double R = (B.hmax > h_i) ? B.hmax : h_i;
                for_each_candidate(B.grid, xs, R, visit, h_i);
            }
            // the partly filled last chunk (entries past `listed` are never read)
            if (G == 1 && list_row && listed < a.list.cap && (listed & (kListChunk - 1)))
                flush_list_chunk(stage, list_row + (listed & ~(kListChunk - 1)));
        } else if ((m_i > 0) && (rho_i > 0)) {
            listed = a.list.cap + 1;  // the force loop still runs for i: send it to the scan
        }
        if constexpr (G > 1) {
            gr0 = group_sum<G>(gr0); gr1 = group_sum<G>(gr1); gr2 = group_sum<G>(gr2);
            gp0 = group_sum<G>(gp0); gp1 = group_sum<G>(gp1); gp2 = group_sum<G>(gp2);
            gv00 = group_sum<G>(gv00); gv01 = group_sum<G>(gv01); gv02 = group_sum<G>(gv02);
            gv10 = group_sum<G>(gv10); gv11 = group_sum<G>(gv11); gv12 = group_sum<G>(gv12);
            gv20 = group_sum<G>(gv20); gv21 = group_sum<G>(gv21); gv22 = group_sum<G>(gv22);
            maxd = group_max<G>(maxd);
            mn_r = group_min<G>(mn_r); mx_r = group_max<G>(mx_r);
            mn_p = group_min<G>(mn_p); mx_p = group_max<G>(mx_p);
            mn_v0 = group_min<G>(mn_v0); mx_v0 = group_max<G>(mx_v0);
            mn_v1 = group_min<G>(mn_v1); mx_v1 = group_max<G>(mx_v1);
            mn_v2 = group_min<G>(mn_v2); mx_v2 = group_max<G>(mx_v2);
        }
        GradSums S = {{gr0, gr1, gr2, gp0, gp1, gp2, gv00, gv01, gv02, gv10, gv11, gv12, gv20, gv21, gv22},
                      {mn_r, mn_p, mn_v0, mn_v1, mn_v2}, {mx_r, mx_p, mx_v0, mx_v1, mx_v2}, maxd};
        finish_gradients(a, i, xi, ri, S, g_out, f_out);
        if (a.list.idx && sub == 0) a.list.count[t] = listed;
    });
    if constexpr (G == 1) {
        wave_store_records(stage, a.grad, 15, out_i, valid, g_out);
        if (a.frec_out) {
            const ForceRec &r = f_out;
            const double w[sizeof(ForceRec) / 8] = {
                r.v[0], r.v[1], r.v[2], r.h, r.hinv, r.rho, r.P, r.cs, r.V, r.dhsml, r.fce, r.nvt[0], r.nvt[1], r.nvt[2],
                r.nvt[3], r.nvt[4], r.nvt[5], r.gr[0], r.gr[1], r.gr[2], r.gp[0], r.gp[1], r.gp[2], r.gv[0], r.gv[1],
                r.gv[2], r.gv[3], r.gv[4], r.gv[5], r.gv[6], r.gv[7], r.gv[8], r.cn, r.e};
            wave_store_records(stage, reinterpret_cast<double *>(a.frec_out), sizeof(ForceRec) / 8, out_i, valid, w);
        }
    } else if (valid && sub == 0) {
        for (int k = 0; k < 15; k++) a.grad[15 * (size_t)out_i + k] = g_out[k];
        if (a.frec_out) a.frec_out[out_i] = f_out;
    }
    if (a.list.idx) {
        // wavefronts with a particle of more than cap neighbours
        const bool over = __any(listed > a.list.cap);
        if ((threadIdx.x & 63) == 0 && over) atomicAdd(&ctr_slot(a.ctr)->overflow_slices, 1);
    }
    wave_add_u64(&ctr_slot(a.ctr)->interactions, cnt);
}

// Tree: the particles whose rows do not hold their pair set (`list`, a device
// count; W = 64), or, without rows, every active one (list NULL; W = 16, as there
// are 15 sums: 40 k active of 400 k 0.48 ms, with W = 64 0.64, with one lane each
// 2.6), W lanes each: the lanes share the walk and the pairs' terms.  Each sum is then added up by one
// lane in ascending slot order, the order of the merged rows, so a particle's
// bits do not depend on the rows.  250 k particles in Plummer spheres: row kernel
// and this one 0.60 ms, against 4.2 ms for the row kernel with these particles
// walking in a lane each.
template <int W>
__global__ __launch_bounds__(kBlock) void gradients_walk_kernel(GradientArgs a, const int *list, const int *count)
{
    static_assert(W >= 16, "15 sums");
    __shared__ GroupWalkLds<W> walk[kBlock / W];
    __shared__ double term_lds[kBlock / W][W][8];
    const int lane = (int)threadIdx.x % W;
    double (*term)[8] = term_lds[threadIdx.x / W];
    const int n = list ? *count : a.n_active;
    const int n_groups = (int)(gridDim.x * (kBlock / W));
    const int q_a = lane % 3, q_b = 3 + min(lane / 3, 4);  // lane < 15: the sum of w[q_a] d[q_b - 3]
    unsigned long long cnt = 0;
    bool over = false;
    for (int u = (int)(blockIdx.x * kBlock + threadIdx.x) / W; u < n; u += n_groups) {
        const int t = list ? list[u] : u;
        const int i = a.active[t];
        const BoxDesc &B = a.boxes[a.box_of[i]];
        const GradRec ri = a.rec[i];
        const double4 xi = a.xh[i];
        const double h_i = xi.w, rho_i = ri.vr.w, p_i = ri.pm.x, m_i = ri.pm.y;
        int *list_row = a.list.idx ? a.list.idx + (size_t)t * a.list.cap : nullptr;
        int listed = 0;
        GradSums S = {};
        if ((m_i > 0) && (rho_i > 0) && (h_i > 0)) {  // GasGrad_isactive (gradients.c:66-75)
            double hinv, hinv3, hinv4, sum = 0;
            kernel_hinv(h_i, hinv, hinv3, hinv4);
            const double h2_i = h_i * h_i;
            const double xs[3] = {xi.x, xi.y, xi.z};
            group_tree_walk<W, true>(a.tree, B, xs, h_i, h_i, lane, walk[threadIdx.x / W], [&](int j, bool valid) {
                double dp[3] = {0, 0, 0}, r2 = 0;
                double4 xj = make_double4(0, 0, 0, 0), vr = xj;
                double2 pm = make_double2(0, 0);
                if (valid) {
                    xj = a.xh[j];
                    dp[0] = xs[0] - xj.x;
                    dp[1] = xs[1] - xj.y;
                    dp[2] = xs[2] - xj.z;
                    wrap_dp(B.box, dp);
                    r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                    valid = r2 > 0 && !((r2 >= h2_i) && (r2 >= xj.w * xj.w));
                }
                if (valid) {
                    vr = a.rec[j].vr;
                    pm = a.rec[j].pm;
                    valid = (pm.y > 0) && (vr.w > 0);
                }
                const uint64_t below = (1ull << lane) - 1, pairs = group_ballot<W>(valid);
                const int k = listed + __popcll(pairs & below);
                if (valid && list_row && k < a.list.cap) list_row[k] = j;
                listed += __popcll(pairs);
                if (!(xj.w > 0)) valid = false;
                const double r = sqrt(r2);
                if (valid) {
                    cnt++;
                    if (r > S.maxd) S.maxd = r;
                }
                const double d[5] = {vr.w - rho_i, pm.x - p_i, vr.x - ri.vr.x, vr.y - ri.vr.y, vr.z - ri.vr.z};
                if (valid)
                    for (int q = 0; q < 5; q++) minmax_check(d[q], S.mn[q], S.mx[q]);
                const bool inside = valid && r < h_i;
                const uint64_t in = group_ballot<W>(inside);
                if (inside) {
                    const double wk_i = kernel_w(r * hinv, hinv3);
                    double *o = term[__popcll(in & below)];
                    for (int q = 0; q < 3; q++) o[q] = -wk_i * dp[q];
                    for (int q = 0; q < 5; q++) o[3 + q] = d[q];
                }
                wave_lds_fence();
                const int n_in = __popcll(in);
#pragma unroll 4
                for (int p = 0; p < n_in; p++) sum += term[p][q_a] * term[p][q_b];
                wave_lds_fence();
            });
#pragma unroll
            for (int q = 0; q < 15; q++) S.g[q] = __shfl(sum, q, W);
            S.maxd = group_max<W>(S.maxd);
            for (int q = 0; q < 5; q++) {
                S.mn[q] = group_min<W>(S.mn[q]);
                S.mx[q] = group_max<W>(S.mx[q]);
            }
        } else if ((m_i > 0) && (rho_i > 0)) {
            listed = a.list.cap + 1;  // as in gradients_kernel
        }
        double g_out[15];
        ForceRec f_out;
        finish_gradients(a, i, xi, ri, S, g_out, f_out);
        if (lane == 0) {
            for (int k = 0; k < 15; k++) a.grad[15 * (size_t)i + k] = g_out[k];
            if (a.frec_out) a.frec_out[i] = f_out;
            if (a.list.idx) a.list.count[t] = listed;
        }
        over |= listed > a.list.cap;
    }
    if (a.list.idx && lane == 0 && over) atomicAdd(&ctr_slot(a.ctr)->overflow_slices, 1);
    wave_add_u64(&ctr_slot(a.ctr)->interactions, cnt);
}

// ---------------------------------------------------------------------------
// force (hydro_evaluate.h:22-516, hydro_core_meshless.h, compute_finitevol_faces.h,
// final operations hydro_toplevel.c:652-767)
// ---------------------------------------------------------------------------
__global__ void pack_force_kernel(int n, const double4 *posm, const double4 *velu, const double *hsml,
                                  const double *rho, const double *pres, const double *dhsml, const double *cn,
                                  const double *fce, const double *nvt, const double *grad, double gamma,
                                  ForceRec *rec)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    rec[k] = make_force_rec(posm[k], velu[k], rho[k], pres[k], hsml[k], dhsml[k], cn[k], fce[k], nvt + 6 * (size_t)k,
                            grad + 15 * (size_t)k, gamma);
}


// The force loop over the pair lists (lists of <= 64): pairs that reach the
// exact Riemann solver (or the KT flux of a failed estimate) are left to
// force_deferred_kernel and added by force_finish_kernel, after all other pairs
// of the particle; particles whose list overflowed are left to
// force_wave_fp64_kernel.
// Bounded by the latency of the pair's serial arithmetic at two wavefronts per
// SIMD (vector units 64 % busy; a third would need the records of its 64 pairs
// in 13 KB of LDS).  33 k particles: 61 us against 145 us with one lane per
// particle; 2.1 M: 3.43 against 3.38 ms.
__global__ __launch_bounds__(64, 2) void force_list_kernel(ForceArgs a)
{
    __shared__ PairLoopLds<ForceRec> lds;
    const int lane = threadIdx.x, sub = lane % kForceLanes;
    const int t = xcd_block() * (64 / kForceLanes) + lane / kForceLanes;
    bool valid = t < a.n_active;
    int n = 0, i = 0;
    if (valid) {
        n = a.list.count[t];
        i = a.active[t];
        if (n > a.list.cap) {  // evaluated by the wavefront loop for long pair sets
            if (sub == 0) {
                a.defer.count[t] = 0;
                a.defer.raw[t] = 0;
            }
            valid = false;
        }
    }
    const double4 pi = a.posm[i];
    const double rho_i = a.rec[i].rho, cs_i = a.rec[i].cs;
    const bool live = valid && (pi.w > 0) && (rho_i > 0);
    if (!live) n = 0;
    const BoxInfo &box = a.boxes[a.box_of[i]].box;
    const double L[3] = {box.L[0], box.L[1], box.L[2]};
    double acc[3] = {0, 0, 0}, dte = 0, out_vsig = cs_i;
    int status = 0, n_deferred = 0;
    uint64_t dmask = 0;
    unsigned long long cnt = 0;
    ROut<double> ro = {0, 0, {0, 0, 0}, 0};
    pair_list_loop(lds, a.rec, a.posm, a.list.idx + (size_t)t * a.list.cap, n, i,
                   [&](const ForceRec &I, const ForceRec &J, const double4 &xj, int j, int k) {
        double dp[3] = {pi.x - xj.x, pi.y - xj.y, pi.z - xj.z};
#pragma unroll
        for (int c = 0; c < 3; c++) dp[c] = wrap_axis(dp[c], L[c], 0.5 * L[c]);
        const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
        double Fv[3], Fp, vsig;
        int mask;
        const int e = force_pair<double, true, false, true>(I, J, dp, r2, a.G, ro, Fv, Fp, vsig, mask);
        cnt++;
        if (e == kDeferred) {
            dmask |= 1ull << k;
            n_deferred++;
            return;
        }
        if (e > status) status = e;
        acc[0] += Fv[0];
        acc[1] += Fv[1];
        acc[2] += Fv[2];
        dte += Fp;
        if (vsig > out_vsig) out_vsig = vsig;
        if (a.is_active && !a.is_active[j]) {
            if (vsig > kWakeup * a.vsig_old[j]) a.wakeup[j] = 1;  // WAKEUP (hydro_evaluate.h:485-495)
        }
    });
    if (status) atomicMax(&ctr_slot(a.ctr)->status, status);
    for (int c = 0; c < 3; c++) acc[c] = group_sum<kForceLanes>(acc[c]);
    dte = group_sum<kForceLanes>(dte);
    out_vsig = group_max<kForceLanes>(out_vsig);
    dmask = group_or<kForceLanes>(dmask);
    n_deferred = group_sum_int<kForceLanes>(n_deferred);
    if (valid && sub == 0) {
        if (live) {
            // raw sums: finished by force_finish_kernel after the deferred pairs
            a.defer.mask[t] = dmask;
        } else {
            if (pi.w > 0) dte /= pi.w;
            out_vsig = kMinReal;
        }
        a.defer.count[t] = n_deferred;
        a.defer.raw[t] = live ? 1 : 0;
        a.acc[3 * (size_t)i + 0] = acc[0];
        a.acc[3 * (size_t)i + 1] = acc[1];
        a.acc[3 * (size_t)i + 2] = acc[2];
        a.dtu[i] = dte;
        a.vsig[i] = out_vsig;
    }
    wave_add_u64(&ctr_slot(a.ctr)->interactions, cnt);
}

// One lane's force loop where no list of at most 64 pairs holds the set.
// USE_LIST: walk the pair list written by the gradient kernel (particles that
// overflowed it are skipped and left to force_wave_fp64_kernel); otherwise scan
// the grid or tree (no list: every particle).  Pairs that reach the exact
// Riemann solver are summed after all other pairs of the particle, in a second
// walk over the pairs.
template <bool USE_LIST>
__global__ __launch_bounds__(kBlock) void force_kernel(ForceArgs a)
{
    extern __shared__ double part_lds[];
    const int t = xcd_block() * (int)blockDim.x + threadIdx.x;
    bool valid = t < a.n_active;
    if (USE_LIST && valid && a.list.count[t] > a.list.cap) valid = false;
    unsigned long long cnt = 0, nretry = 0, nexact = 0;
    for_box(a.boxes, a.box_of, valid ? a.active[t] : 0, valid, [&](const BoxDesc &G) {
        const int i = a.active[t];
        const double4 pi = a.posm[i];
        double acc[3] = {0, 0, 0}, dte = 0, vmax = kMinReal;
        const double m_i = pi.w;
        const ForceRec I = a.rec[i];
        int status = 0;
        if ((m_i > 0) && (I.rho > 0)) {
            const double x_i[3] = {pi.x, pi.y, pi.z};
            double out_vsig = I.cs;
            ROut<double> ro = {0, 0, {0, 0, 0}, 0};
            const double h2_i = I.h * I.h;
            int n_deferred = 0, k_pair = 0;
            LaneSums part(part_lds);
            auto add = [&](int lane, int j, const double Fv[3], double Fp, double vsig, int mask, int e) {
                if (e > status) status = e;
                nretry += (mask & 8) ? 1 : 0;
                nexact += (mask & 4) ? 1 : 0;
                const double v[4] = {Fv[0], Fv[1], Fv[2], Fp};
                part.add(lane, v);
                if (vsig > out_vsig) out_vsig = vsig;
                if (a.is_active && !a.is_active[j]) {
                    if (vsig > kWakeup * a.vsig_old[j]) a.wakeup[j] = 1;  // WAKEUP (hydro_evaluate.h:485-495)
                }
            };
            // pass 0: every pair but the deferred ones; pass 1: only those
            auto visit = [&](int j, bool check, int pass) {
                const double4 xj = a.posm[j];
                double dp[3] = {x_i[0] - xj.x, x_i[1] - xj.y, x_i[2] - xj.z};
                wrap_dp(G.box, dp);
                const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                const ForceRec J = a.rec[j];
                if (check) {
                    if ((r2 >= h2_i) && (r2 >= J.h * J.h)) return;
                    if (r2 <= 0) return;
                    if (!(xj.w > 0) || !(J.rho > 0)) return;  // hydro_evaluate.h:149-150
                }
                double Fv[3], Fp, vsig;
                int mask;
                const int e = force_pair<double, true>(I, J, dp, r2, a.G, ro, Fv, Fp, vsig, mask);
                if (pass == 0) {
                    cnt++;
                    const int k = k_pair++;
                    if (e == kDeferred) {
                        n_deferred++;
                        return;
                    }
                    add(k % kForceLanes, j, Fv, Fp, vsig, mask, e);
                } else if (e == kDeferred) {
                    const int e2 = force_pair<double, false>(I, J, dp, r2, a.G, ro, Fv, Fp, vsig, mask);
                    add(0, j, Fv, Fp, vsig, mask, e2);
                }
            };
            for (int pass = 0; pass < 2; pass++) {
                if (pass == 1) {
                    part.fold();
                    if (n_deferred == 0) break;
                }
                if (USE_LIST) {
                    // the list holds the pair set in the gradient kernel's scan order,
                    // which is this kernel's scan order as well (same predicate, same R)
                    const int n = a.list.count[t];
                    const int *row = a.list.idx + (size_t)t * a.list.cap;
                    for (int k = 0; k < n; k++) visit(row[k], false, pass);
                } else {
                    for_each_neighbour_candidate(a.tree, G, x_i, I.h, true, [&](int j) { visit(j, true, pass); });
                }
            }
            for (int c = 0; c < 3; c++) acc[c] = part.total(c);
            dte = part.total(3);
            if (vmax < out_vsig) vmax = out_vsig;
            force_final_ops(acc, dte, I.v, m_i, I.h, a.max_hsml);
        } else if (m_i > 0) {
            dte /= m_i;
        }
        a.acc[3 * (size_t)i + 0] = acc[0];
        a.acc[3 * (size_t)i + 1] = acc[1];
        a.acc[3 * (size_t)i + 2] = acc[2];
        a.dtu[i] = dte;
        a.vsig[i] = vmax;
        if (status) atomicMax(&ctr_slot(a.ctr)->status, status);
    });
    wave_add_u64(&ctr_slot(a.ctr)->interactions, cnt);
    wave_add_u64(&ctr_slot(a.ctr)->retries, nretry);
    wave_add_u64(&ctr_slot(a.ctr)->exact_calls, nexact);
}

// Deferred pairs q in [q_begin, min(total, q_end)): one pair per lane, with
// the exact Riemann solver.
__global__ __launch_bounds__(kBlock) void force_deferred_kernel(ForceArgs a)
{
    const int q = a.defer.q_begin + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int q_end = min(*a.defer.total, a.defer.q_end);
    const bool valid = q < q_end;
    const int2 ij = valid ? a.defer.pair[q - a.defer.q_begin] : make_int2(0, 0);
    unsigned long long nretry = 0, nexact = 0;
    for_box(a.boxes, a.box_of, ij.x, valid, [&](const BoxDesc &G) {
        const int i = ij.x, j = ij.y;
        const ForceRec I = a.rec[i], J = a.rec[j];
        const double4 pi = a.posm[i], xj = a.posm[j];
        double dp[3] = {pi.x - xj.x, pi.y - xj.y, pi.z - xj.z};
        wrap_dp(G.box, dp);
        const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
        ROut<double> ro = {0, 0, {0, 0, 0}, 0};
        double Fv[3], Fp, vsig;
        int mask;
        const int e = force_pair<double, false, true>(I, J, dp, r2, a.G, ro, Fv, Fp, vsig, mask);
        nretry += (mask & 8) ? 1 : 0;
        nexact += (mask & 4) ? 1 : 0;
        double *o = a.defer.result + 5 * (size_t)(q - a.defer.q_begin);
        o[0] = Fv[0]; o[1] = Fv[1]; o[2] = Fv[2]; o[3] = Fp; o[4] = vsig;
        if (a.is_active && !a.is_active[j]) {
            if (vsig > kWakeup * a.vsig_old[j]) a.wakeup[j] = 1;
        }
        if (e) atomicMax(&ctr_slot(a.ctr)->status, e);
    });
    wave_add_u64(&ctr_slot(a.ctr)->retries, nretry);
    wave_add_u64(&ctr_slot(a.ctr)->exact_calls, nexact);
}

// Add the deferred pairs of this round to the raw sums (in list order) and,
// for particles whose deferred pairs are all in, apply the final operations.
// `velu` and `hsml` give the FP64 velocity and hsml of i.
__global__ __launch_bounds__(kBlock) void force_finish_kernel(ForceArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n_active || !a.defer.raw[t]) return;
    const int i = a.active[t];
    double acc[3] = {a.acc[3 * (size_t)i + 0], a.acc[3 * (size_t)i + 1], a.acc[3 * (size_t)i + 2]};
    double dte = a.dtu[i], out_vsig = a.vsig[i];
    const int q0 = a.defer.offset[t], q1 = q0 + a.defer.count[t];
    for (int q = max(q0, a.defer.q_begin); q < min(q1, a.defer.q_end); q++) {
        const double *o = a.defer.result + 5 * (size_t)(q - a.defer.q_begin);
        acc[0] += o[0];
        acc[1] += o[1];
        acc[2] += o[2];
        dte += o[3];
        if (o[4] > out_vsig) out_vsig = o[4];
    }
    if (q1 <= a.defer.q_end) {
        double vmax = kMinReal;
        if (vmax < out_vsig) vmax = out_vsig;
        const double4 v = a.velu[i];
        const double vi[3] = {v.x, v.y, v.z};
        force_final_ops(acc, dte, vi, a.posm[i].w, a.hsml[i], a.max_hsml);
        out_vsig = vmax;
        a.defer.raw[t] = 0;
    }
    a.acc[3 * (size_t)i + 0] = acc[0];
    a.acc[3 * (size_t)i + 1] = acc[1];
    a.acc[3 * (size_t)i + 2] = acc[2];
    a.dtu[i] = dte;
    a.vsig[i] = out_vsig;
}

// neighbour-set sizes for a fixed hsml (same predicates as the stage kernels)
__global__ __launch_bounds__(kBlock) void neighbor_count_kernel(const BoxDesc *boxes, const int *box_of,
                                                                TreeArgs tree, int mode, int n_active,
                                                                const int *active, const double4 *posm,
                                                                const double *hsml, int *counts, Counters *ctr)
{
    const int t = xcd_block() * kBlock + threadIdx.x;
    unsigned long long cnt = 0;
    const bool valid = t < n_active;
    for_box(boxes, box_of, valid ? active[t] : 0, valid, [&](const BoxDesc &G) {
        const int i = active[t];
        const double4 pi = posm[i];
        const double h = hsml[i], h2 = h * h;
        const double xs[3] = {pi.x, pi.y, pi.z};
        for_each_neighbour_candidate(tree, G, xs, h, mode != 0, [&](int j) {
            const double4 pj = posm[j];
            double dp[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
            wrap_dp(G.box, dp);
            const double r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
            if (mode == 0) {
                if (r2 < h2) cnt++;
            } else {
                const double h_j = hsml[j];
                if ((r2 >= h2) && (r2 >= h_j * h_j)) return;
                if (r2 <= 0) return;
                cnt++;
            }
        });
        if (counts) counts[t] = (int)cnt;
    });
    wave_add_u64(&ctr_slot(ctr)->interactions, cnt);
}

inline unsigned nblocks(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }
inline unsigned nblocks(long long n, int block) { return (unsigned)((n + block - 1) / block); }


}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
void launch_cell_keys(hipStream_t s, int n, const double *pos, const BoxDesc *boxes, const int *box_caller,
                      uint64_t *keys, int *iota)
{
    if (n > 0) hipLaunchKernelGGL(cell_keys_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, pos, boxes, box_caller, keys, iota);
}
void launch_gather_sorted(hipStream_t s, int n, const int *perm, const double *pos, const double *vel,
                          const double *mass, const double *u, const BoxDesc *boxes, const int *box_caller,
                          double4 *posm, double4 *velu, float4 *posf, int *inv, int *box_of)
{
    if (n > 0)
        hipLaunchKernelGGL(gather_sorted_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, perm, pos, vel, mass, u, boxes,
                           box_caller, posm, velu, posf, inv, box_of);
}
void launch_gather_scalar(hipStream_t s, int n, const int *perm, const double *src, double *dst, int width)
{
    if (((long long)n * width) > 0) hipLaunchKernelGGL(gather_scalar_kernel, dim3(nblocks((long long)n * width)), dim3(kBlock), 0, s, n, perm, src,
                       dst, width);
}
void launch_export(hipStream_t s, ExportArgs &a)
{
    unsigned blocks = 0;
    for (int q = 0; q < a.n_fields; q++) {
        a.first_block[q] = blocks;
        blocks += nblocks((long long)a.n * a.field[q].w);
    }
    if (blocks > 0) hipLaunchKernelGGL(export_kernel, dim3(blocks), dim3(kBlock), 0, s, a);
}
void launch_export_u8(hipStream_t s, int n, const int *inv, const uint8_t *src, uint8_t *dst)
{
    if (n > 0) hipLaunchKernelGGL(export_u8_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, inv, src, dst);
}
void launch_fill_fields(hipStream_t s, const FillArgs &a)
{
    if (a.n > 0 && a.n_fills > 0) hipLaunchKernelGGL(fill_fields_kernel, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
}
void launch_iota(hipStream_t s, int n, int *p)
{
    if (n > 0) hipLaunchKernelGGL(iota_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, p);
}
void launch_restore(hipStream_t s, int n, double *hsml, const double *hsml0, double *cn, const double *cn0, double *vsig,
                    const double *vsig0, double *dmass, const double *dmass0)
{
    if (n > 0)
        hipLaunchKernelGGL(restore_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, hsml, hsml0, cn, cn0, vsig, vsig0,
                           dmass, dmass0);
}
void launch_publish_counters(hipStream_t s, const Counters *ctr, Counters *host)
{
    hipLaunchKernelGGL(publish_counters_kernel, dim3(1), dim3(kCtrSpread), 0, s, ctr, host);
}
void launch_cell_ranges(hipStream_t s, int n, const double4 *posm, const BoxDesc *boxes, const int *box_of,
                        int2 *range, int ncell)
{
    if ((2LL * ncell) > 0) hipLaunchKernelGGL(fill_int_kernel, dim3(nblocks(2LL * ncell)), dim3(kBlock), 0, s, (int *)range, 2 * ncell, 0);
    if (n > 0) hipLaunchKernelGGL(cell_ranges_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, posm, boxes, box_of, range);
}
void launch_pair_prepare(hipStream_t s, PairPrepareArgs &a, int n_boxes, Counters *ctr)
{
    if (n_boxes > 0 || ctr)
        hipLaunchKernelGGL(clear_box_hmax_kernel, dim3(nblocks(std::max(n_boxes, 1))), dim3(kBlock), 0, s, n_boxes, a.boxes,
                           ctr);
    a.cell_blocks = (int)nblocks(a.n_cells);
    const unsigned blocks = a.n_tiles + a.cell_blocks + (a.rec ? nblocks(a.n) : 0);
    if (blocks > 0) hipLaunchKernelGGL(pair_prepare_kernel, dim3(blocks), dim3(kBlock), 0, s, a);
}
void launch_flag_unconverged(hipStream_t s, const int *n_live_dev, Counters *ctr)
{
    hipLaunchKernelGGL(flag_unconverged_kernel, dim3(1), dim3(64), 0, s, n_live_dev, ctr);
}
void launch_clear_counters(hipStream_t s, Counters *ctr)
{
    hipLaunchKernelGGL(clear_counters_kernel, dim3(1), dim3(kCtrSpread), 0, s, ctr);
}
void launch_map_active(hipStream_t s, int n_active, const int *active_caller, const int *inv, int *active_sorted)
{
    if ((n_active) > 0) hipLaunchKernelGGL(map_active_kernel, dim3(nblocks(n_active)), dim3(kBlock), 0, s, n_active, active_caller, inv,
                       active_sorted);
}
void launch_density_begin(hipStream_t s, Counters *ctr, int *counts)
{
    hipLaunchKernelGGL(density_begin_kernel, dim3(1), dim3(kCtrSpread), 0, s, ctr, counts);
}
void launch_density_init(hipStream_t s, int n_active, const int *active, const double4 *posm, double *hsml, double *left,
                         double *right, double max_hsml, int *live_flag)
{
    if ((n_active) > 0) hipLaunchKernelGGL(density_init_kernel, dim3(nblocks(n_active)), dim3(kBlock), 0, s, n_active, active, posm,
                       hsml, left, right, max_hsml, live_flag);
}
void launch_edge_reset(hipStream_t s, int cap, const int *n_edge, const int *edge_list, const double *hsml_entry,
                       double *hsml, double *left, double *right, int *iter)
{
    if (cap > 0)
        hipLaunchKernelGGL(edge_reset_kernel, dim3(nblocks(cap)), dim3(kBlock), 0, s, cap, n_edge, edge_list,
                           hsml_entry, hsml, left, right, iter);
}
void launch_density_finalize(hipStream_t s, int n_active, const int *active, const double4 *posm,
                             const double4 *velu, const double *hsml, double *num_ngb, double *rho, double *pres,
                             double gm1)
{
    if ((n_active) > 0) hipLaunchKernelGGL(density_finalize_kernel, dim3(nblocks(n_active)), dim3(kBlock), 0, s, n_active, active, posm,
                       velu, hsml, num_ngb, rho, pres, gm1);
}
void launch_sym_rows(hipStream_t s, const SymRowArgs &a)
{
    if (a.n <= 0) return;
    launch_fill_int(s, a.bcount, a.n, 0);
    launch_fill_int(s, a.wcount, 2, 0);
    hipLaunchKernelGGL(sym_rows_scatter_kernel, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
    hipLaunchKernelGGL(sym_rows_wave_kernel, dim3(2048), dim3(kBlock), 0, s, a);
    hipLaunchKernelGGL(sym_rows_sort_kernel, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a.n, a.brow, a.bcount);
}
template <GradSource SRC>
static void launch_gradients_from(hipStream_t s, const GradientArgs &a, dim3 grid, dim3 block)
{
    if (a.block == 64) hipLaunchKernelGGL((gradients_kernel<64, SRC>), grid, block, 0, s, a);
    else if (a.block == 128) hipLaunchKernelGGL((gradients_kernel<128, SRC>), grid, block, 0, s, a);
    else if (a.block == 512) hipLaunchKernelGGL((gradients_kernel<512, SRC>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((gradients_kernel<kBlock, SRC>), grid, block, 0, s, a);
}
void launch_gradients(hipStream_t s, const GradientArgs &a)
{
    if (a.n_active <= 0) return;
    const dim3 grid(nblocks(a.n_active, a.block)), block(a.block);
    if (a.lanes == 8) {
        const dim3 few(nblocks(8LL * a.n_active));
        if (a.dcache_idx) hipLaunchKernelGGL((gradients_kernel<kBlock, kFromGridRows, 8>), few, dim3(kBlock), 0, s, a);
        else hipLaunchKernelGGL((gradients_kernel<kBlock, kFromWalk, 8>), few, dim3(kBlock), 0, s, a);
    } else if (a.tree.nodes) {
        // the list's length is on the device: at most what fills the chip
        if (a.brow) {
            const dim3 waves(std::min(2048u, nblocks(64LL * a.n_active)));
            launch_gradients_from<kFromTreeRows>(s, a, grid, block);
            hipLaunchKernelGGL(gradients_walk_kernel<64>, waves, dim3(kBlock), 0, s, a, a.far_list, a.n_far);
        } else {
            const dim3 groups(nblocks(16LL * a.n_active));
            hipLaunchKernelGGL(gradients_walk_kernel<16>, groups, dim3(kBlock), 0, s, a, nullptr, nullptr);
        }
    } else if (a.dcache_idx) {
        launch_gradients_from<kFromGridRows>(s, a, grid, block);
    } else {
        launch_gradients_from<kFromWalk>(s, a, grid, block);
    }
}
void launch_pack_force(hipStream_t s, int n, const double4 *posm, const double4 *velu, const double *hsml,
                       const double *rho, const double *pres, const double *dhsml, const double *cn,
                       const double *fce, const double *nvt, const double *grad, double gamma, ForceRec *rec)
{
    if ((n) > 0) hipLaunchKernelGGL(pack_force_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, n, posm, velu, hsml, rho, pres,
                       dhsml, cn, fce, nvt, grad, gamma, rec);
}
void launch_force(hipStream_t s, const ForceArgs &a)
{
    if (a.n_active <= 0) return;
    const int b = min(a.block, kBlock);
    const dim3 grid(nblocks(a.n_active, b)), block(b);
    if (a.list.idx && a.defer.mask)
        hipLaunchKernelGGL(force_list_kernel, dim3(nblocks((long long)kForceLanes * a.n_active, 64)), dim3(64), 0, s, a);
    else if (a.list.idx) hipLaunchKernelGGL(force_kernel<true>, grid, block, part_bytes(b), s, a);
    else hipLaunchKernelGGL(force_kernel<false>, grid, block, part_bytes(b), s, a);
}
namespace {

// exclusive sums of up to kOneBlockScan counts, by one workgroup
__global__ __launch_bounds__(1024) void defer_scan_kernel(int n, const int *count, int *offset)
{
    __shared__ int total[16];
    const int per = (n + 1023) / 1024, lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const int beg = min(per * (int)threadIdx.x, n), end = min(beg + per, n);
    int own = 0;
    for (int k = beg; k < end; k++) own += count[k];
    int sum = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(sum, off, 64);
        if (lane >= off) sum += o;
    }
    if (lane == 63) total[wave] = sum;
    __syncthreads();
    int at = sum - own;
    for (int w = 0; w < wave; w++) at += total[w];
    for (int k = beg; k < end; k++) {
        const int c = count[k];
        offset[k] = at;
        at += c;
    }
}

// one thread per active entry: its deferred pairs q = offset + r (r-th set
// bit k of its mask) that fall in the round get their particle and neighbour
// (i, list entry k), so that the pair kernel starts from both records' indices
__global__ __launch_bounds__(kBlock) void defer_owners_kernel(ForceArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n_active) return;
    const int c = a.defer.count[t];
    if (t == a.n_active - 1) {
        const int total = a.defer.offset[t] + c;
        *a.defer.total = total;
        atomicMax(&a.ctr->deferred, total);  // a graph's passes: the most of any
    }
    if (c == 0) return;
    const int q0 = a.defer.offset[t];
    if (q0 >= a.defer.q_end || q0 + c <= a.defer.q_begin) return;
    uint64_t m = a.defer.mask[t];
    for (int r = 0; r < c && m; r++) {
        const int k = __builtin_ctzll(m);
        m &= m - 1;
        const int q = q0 + r;
        if (q >= a.defer.q_begin && q < a.defer.q_end)
            a.defer.pair[q - a.defer.q_begin] = make_int2(a.active[t], a.list.idx[(size_t)t * a.list.cap + k]);
    }
}

}  // namespace

void launch_defer_scan(hipStream_t s, int n, const int *count, int *offset)
{
    hipLaunchKernelGGL(defer_scan_kernel, dim3(1), dim3(1024), 0, s, n, count, offset);
}
void launch_defer_owners(hipStream_t s, const ForceArgs &a)
{
    if (a.n_active > 0) hipLaunchKernelGGL(defer_owners_kernel, dim3(nblocks(a.n_active)), dim3(kBlock), 0, s, a);
}

void launch_force_deferred(hipStream_t s, const ForceArgs &a, int n_pairs)
{
    if (n_pairs > 0) hipLaunchKernelGGL(force_deferred_kernel, dim3(nblocks(n_pairs)), dim3(kBlock), 0, s, a);
}
void launch_force_finish(hipStream_t s, const ForceArgs &a)
{
    if (a.n_active > 0) hipLaunchKernelGGL(force_finish_kernel, dim3(nblocks(a.n_active)), dim3(kBlock), 0, s, a);
}
void launch_density_heavy(hipStream_t s, const DensitySweepArgs &a, int max_entries)
{
    if (max_entries <= 0) return;
    // up to 2048 workgroups of 4 wavefronts stride over the entries
    const long long blocks = ((long long)max_entries + 3) / 4;
    const dim3 grid((unsigned)(blocks < 2048 ? blocks : 2048));
    hipLaunchKernelGGL(density_heavy_kernel, grid, dim3(kBlock), 0, s, a);
}

void launch_neighbor_counts(hipStream_t s, const BoxDesc *boxes, const int *box_of, const TreeArgs &tree, int mode,
                            int n_active, const int *active, const double4 *posm, const double *hsml, int *counts,
                            Counters *ctr)
{
    if (n_active > 0)
        hipLaunchKernelGGL(neighbor_count_kernel, dim3(nblocks(n_active)), dim3(kBlock), 0, s, boxes, box_of, tree,
                           mode, n_active, active, posm, hsml, counts, ctr);
}
void launch_fill_int(hipStream_t s, int *p, int n, int value)
{
    if ((n) > 0) hipLaunchKernelGGL(fill_int_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n, value);
}
void launch_fill_u8(hipStream_t s, uint8_t *p, int n, uint8_t value)
{
    if ((n) > 0) hipLaunchKernelGGL(fill_u8_kernel, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n, value);
}
void launch_set_flags(hipStream_t s, int n_active, const int *active, uint8_t *flags)
{
    if ((n_active) > 0) hipLaunchKernelGGL(set_flags_kernel, dim3(nblocks(n_active)), dim3(kBlock), 0, s, n_active, active, flags);
}

}  // namespace gzm
