// Single scattering from tabulated two-leg signals (PairTables, src/feffgpu/exafs/forward.py:178-320): the histogram
// of absorber-neighbor distances on the tables' grid r0 + i dr (linear-interpolation weights, minimum image of the
// cell, pairs within rmax, self excluded) and its adjoint in the positions.
//
// The histogram is accumulated in 64-bit fixed point (units of 2^-32 of a pair): integer atomics are associative, so
// the result does not depend on the order the pairs arrive in, and each pair adds exactly 2^32 over its two bins. A
// bin holds up to 2^31 pairs before the signed 64-bit value overflows (the host splits larger calls). The
// adjoint needs no atomics: a wavefront sums an atom's pairs, as absorber and as neighbor, over its lanes and adds the
// lanes in a fixed order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include "fm_device.h"

int fm_set_err(int code, const char *msg);

namespace {

constexpr int PH_THREADS = 256;
constexpr double PH_ONE = 4294967296.0;   // 2^32

// minimum image of v (src/feffgpu/cell.py:26-35): cubic v - L rint(v / L), general cell by fractional rounding
__device__ __forceinline__ void min_image(double (&v)[3], const fm_pair_grid &g) {
    if (g.cell_kind == 1) {
        const double L = g.cell[0];
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] -= L * rint(v[c] / L);
    } else if (g.cell_kind == 2) {
        double f[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) f[c] = v[0] * g.cellinv[0 * 3 + c] + v[1] * g.cellinv[1 * 3 + c] + v[2] * g.cellinv[2 * 3 + c];
#pragma unroll
        for (int c = 0; c < 3; ++c) f[c] -= rint(f[c]);
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = f[0] * g.cell[0 * 3 + c] + f[1] * g.cell[1 * 3 + c] + f[2] * g.cell[2 * 3 + c];
    }
}

// Pair (a, j): displacement j - a (minimum image) and distance; false outside rmax or for coincident atoms
// (r^2 <= 1e-6, as forward.py:259, 292 exclude the atom itself).
__device__ __forceinline__ bool pair(const double *pa, const double *pj, const fm_pair_grid &g, double (&v)[3], double &r) {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = pj[c] - pa[c];
    min_image(v, g);
    const double r2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    if (!(r2 <= g.rmax * g.rmax) || !(r2 > 1e-6)) return false;
    r = sqrt(r2);
    return true;
}

// lower bin and upper weight of distance r (forward.py:264-266, 296-298): u = (r - r0) / dr, i0 = floor(u) clamped
// to 0..nr-2, f = u - i0 clamped to [0, 1]; dfdr: d f / d r (1 / dr inside the clamp, else 0)
__device__ __forceinline__ void bin_of(double r, const fm_pair_grid &g, int &i0, double &f, double &dfdr) {
    const double u = (r - g.r0) / g.dr;
    double fl = floor(u);
    fl = fl < 0.0 ? 0.0 : (fl > g.nr - 2 ? (double)(g.nr - 2) : fl);
    i0 = (int)fl;
    f = u - fl;
    dfdr = (f >= 0.0 && f <= 1.0) ? 1.0 / g.dr : 0.0;
    f = f < 0.0 ? 0.0 : (f > 1.0 ? 1.0 : f);
}

__global__ __launch_bounds__(PH_THREADS) void k_pair_hist(int natom, const double *pos, int nabs, const int32_t *absorbers,
                                                           const int32_t *ipot, int npot, fm_pair_grid g,
                                                           unsigned long long *hist, int32_t *nshort) {
    __shared__ int cnt[PH_THREADS / FM_WAVE];
    const int c = blockIdx.y, ai = blockIdx.x;
    const int a = absorbers ? absorbers[ai] : ai;
    if (a < 0 || a >= natom) return;           // an absorber index outside the configuration adds nothing
    const double *P = pos + (size_t)c * natom * 3;
    const double pa[3] = {P[3 * a], P[3 * a + 1], P[3 * a + 2]};
    int shorts = 0;
    for (int j = threadIdx.x; j < natom; j += PH_THREADS) {
        double v[3], r;
        if (!pair(pa, P + 3 * (size_t)j, g, v, r)) continue;
        if (r < g.r0) ++shorts;
        const int p = ipot[j];
        if (p < 0 || p >= npot) continue;
        int i0;
        double f, dfdr;
        bin_of(r, g, i0, f, dfdr);
        const unsigned long long up = (unsigned long long)llrint(f * PH_ONE);
        unsigned long long *h = hist + (size_t)p * g.nr + i0;
        atomicAdd(h, (unsigned long long)PH_ONE - up);
        atomicAdd(h + 1, up);
    }
    if (nshort) {
        for (int off = FM_WAVE / 2; off > 0; off >>= 1) shorts += __shfl_xor(shorts, off, FM_WAVE);
        if ((threadIdx.x & (FM_WAVE - 1)) == 0) cnt[threadIdx.x / FM_WAVE] = shorts;
        __syncthreads();
        if (threadIdx.x == 0) {
            int s = 0;
            for (int w = 0; w < PH_THREADS / FM_WAVE; ++w) s += cnt[w];
            if (s) atomicAdd(nshort, s);
        }
    }
}

// ------------------------------------------------------------------------------------------------ candidate pairs
// Most pairs of a configuration lie outside rmax (85 % of a 28.7 A box at 9.4 A), and the exact FP64 distance with its
// three divisions costs about ten times a float32 one. So the kernels below test every pair in float32 first, queue
// the indices of those that may lie within rmax, and evaluate whole wavefronts of queued pairs exactly (pair() above:
// the same FP64 operations on the same positions for every pair that counts).
//
// The float32 test must never drop a pair that the exact one keeps:
//  - periodic cells: fractional coordinates u = f - rint(f), f = pos / L (cubic) or pos cellinv, in FP64 and rounded to
//    float (2^-25 of a cell); differences and their float image: 2e-7 of a cell per component; the threshold allows
//    1e-6 of the cell's summed edges and 1e-5 of rmax. A general cell's components within 1e-5 of half a cell, where
//    float and FP64 may pick different images of different length, always pass (in a cubic cell both images have the
//    same length). Coordinates beyond 1e6 cells become NaN, and NaN always passes.
//  - no cell: displacements from the configuration's first atom in float, the threshold widened by 4e-7 of both
//    atoms' largest component.
struct Cand {
    float x, y, z, m;      // the float coordinates; m: the widening (no cell), else unused
};
struct CandTest {
    float c[9];            // general cell (rows the lattice vectors)
    float rm, thr;         // widened cutoff; its square (cubic: in units of the cell)
};
template <int KIND> __device__ __forceinline__ CandTest cand_test(const fm_pair_grid &g) {
    CandTest t;
    double edges = 0.0;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        t.c[i] = KIND == 2 ? (float)g.cell[i] : 0.f;
        if (KIND == 2) edges += fabs(g.cell[i]);
    }
    if (KIND == 1) edges = 3.0 * g.cell[0];
    const double rm = g.rmax * (1.0 + 1e-5) + 1e-6 * edges;
    t.rm = (float)rm;
    t.thr = (float)(KIND == 1 ? (rm / g.cell[0]) * (rm / g.cell[0]) : rm * rm) * 1.000001f;
    return t;
}
template <int KIND>
__device__ __forceinline__ Cand cand_of(const double *p, const double (&ref)[3], const fm_pair_grid &g) {
    double f[3];
    if (KIND == 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) f[c] = p[c] - ref[c];
        return Cand{(float)f[0], (float)f[1], (float)f[2],
                    4e-7f * (float)fmax(fabs(f[0]), fmax(fabs(f[1]), fabs(f[2])))};
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        f[c] = KIND == 1 ? p[c] / g.cell[0]
                         : p[0] * g.cellinv[c] + p[1] * g.cellinv[3 + c] + p[2] * g.cellinv[6 + c];
        f[c] = fabs(f[c]) < 1e6 ? f[c] - rint(f[c]) : __builtin_nan("");
    }
    return Cand{(float)f[0], (float)f[1], (float)f[2], 0.f};
}
template <int KIND> __device__ __forceinline__ bool cand_pair(const Cand &a, const Cand &j, const CandTest &t) {
    float x = j.x - a.x, y = j.y - a.y, z = j.z - a.z;
    if (KIND == 0) {
        const float w = t.rm + (a.m + j.m);
        return !(x * x + y * y + z * z > w * w);
    }
    x -= rintf(x);
    y -= rintf(y);
    z -= rintf(z);
    if (KIND == 1) return !(x * x + y * y + z * z > t.thr);
    const float h = fmaxf(fabsf(x), fmaxf(fabsf(y), fabsf(z)));
    const float vx = x * t.c[0] + y * t.c[3] + z * t.c[6];
    const float vy = x * t.c[1] + y * t.c[4] + z * t.c[7];
    const float vz = x * t.c[2] + y * t.c[5] + z * t.c[8];
    return !(vx * vx + vy * vy + vz * vz > t.thr) || h > 0.5f - 1e-5f;
}

// The lane's position among the set lanes of a ballot below it.
__device__ __forceinline__ int lanes_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// The histogram with a workgroup's bins in LDS: PH_WAVES wavefronts (a CU's one workgroup, its LDS holds the bins) loop
// over tiles of PH_ROWS absorbers x PH_COLS atoms of a configuration, each wavefront testing its rows against 64 atoms
// at a time and binning its queue of candidates 64 at a time; the grid is at most one workgroup per CU, so the bins
// are cleared and added to hist once per CU however many tiles there are. With every atom an absorber (absorbers
// NULL) only pairs a < j are evaluated and added for both orders: the distance is the same to the bit (differences,
// rint and squares are symmetric), so the integer sums are those of the ordered pairs.
// Bound by the uneven shares of the tiles (256 workgroups are a multiple of the 128 tiles of 2000 atoms, so each gets the
// same tile of every second frame, and those of j <= a are empty): CUs busy 38 %, VALU 25 %. 64 frames x 2000 atoms
// (2.56e8 ordered pairs, 14.7 % within): 0.67 ms; one box of 4000 atoms: 0.041 ms (exact FP64 of every ordered pair, 64
// absorbers per workgroup: 2.00 ms, 0.377 ms).
constexpr int PH_WAVES = 16, PH_ROWS = 128, PH_COLS = 256;

template <int KIND>
__global__ __launch_bounds__(FM_WAVE *PH_WAVES) void k_pair_hist_lds(int natom, int nconf, const double *pos, int nabs,
                                                                     const int32_t *absorbers, const int32_t *ipot,
                                                                     int npot, fm_pair_grid g,
                                                                     unsigned long long *hist, int32_t *nshort) {
    extern __shared__ __align__(16) unsigned long long lh[];
    __shared__ Cand rowc[PH_ROWS], colc[PH_COLS];
    __shared__ int rowi[PH_ROWS];
    __shared__ uint16_t queue[PH_WAVES][2 * FM_WAVE];
    __shared__ int shorts_wg;
    const int t = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(t / FM_WAVE), lane = t % FM_WAVE;
    constexpr int NT = FM_WAVE * PH_WAVES, RW = PH_ROWS / PH_WAVES;
    const int nb = npot * g.nr;
    for (int b = t; b < nb; b += NT) lh[b] = 0ull;
    if (t == 0) shorts_wg = 0;
    const CandTest ct = cand_test<KIND>(g);
    const bool sym = absorbers == nullptr;
    const int ntr = (nabs + PH_ROWS - 1) / PH_ROWS, ntc = (natom + PH_COLS - 1) / PH_COLS;
    const long items = (long)nconf * ntr * ntc;
    uint16_t *const q = queue[wid];
    int shorts = 0;
    for (long it = blockIdx.x; it < items; it += gridDim.x) {
        const int c = (int)(it / ((long)ntr * ntc)), rc = (int)(it - (long)c * ntr * ntc);
        const int r0 = (rc / ntc) * PH_ROWS, c0 = (rc % ntc) * PH_COLS;
        if (sym && c0 + PH_COLS - 1 <= r0) continue;      // uniform: every pair of the tile has j <= a
        const double *P = pos + (size_t)c * natom * 3;
        const double ref[3] = {P[0], P[1], P[2]};
        __syncthreads();                                   // the previous tile (and the cleared bins)
        if (t < PH_ROWS) {
            const int a = r0 + t < nabs ? (sym ? r0 + t : absorbers[r0 + t]) : -1;
            const bool ok = a >= 0 && a < natom;           // an absorber index outside the configuration adds nothing
            rowi[t] = ok ? a : -1;
            rowc[t] = cand_of<KIND>(P + 3 * (size_t)(ok ? a : 0), ref, g);
        } else if (t < PH_ROWS + PH_COLS) {
            const int j = c0 + t - PH_ROWS;
            colc[t - PH_ROWS] = cand_of<KIND>(P + 3 * (size_t)(j < natom ? j : 0), ref, g);
        }
        __syncthreads();
        int head = 0, cnt = 0;
        auto bin = [&](int n) {                            // the first n (<= 64) queued pairs
            fm::wave_sync();
            if (lane < n) {
                const int code = q[(head + lane) & (2 * FM_WAVE - 1)];
                const int a = rowi[code >> 8], j = c0 + (code & 255);
                const double pa[3] = {P[3 * (size_t)a], P[3 * (size_t)a + 1], P[3 * (size_t)a + 2]};
                double v[3], r;
                if (pair(pa, P + 3 * (size_t)j, g, v, r)) {
                    if (r < g.r0) shorts += sym ? 2 : 1;
                    int i0;
                    double f, dfdr;
                    bin_of(r, g, i0, f, dfdr);
                    const unsigned long long up = (unsigned long long)llrint(f * PH_ONE);
                    const unsigned long long lo = (unsigned long long)PH_ONE - up;
                    const int pj = ipot[j], pi = sym ? ipot[a] : -1;
                    const int w = pi == pj ? 2 : 1;        // both orders on the same bins
                    if (pj >= 0 && pj < npot) {
                        atomicAdd(&lh[pj * g.nr + i0], lo * w);
                        atomicAdd(&lh[pj * g.nr + i0 + 1], up * w);
                    }
                    if (w == 1 && pi >= 0 && pi < npot) {
                        atomicAdd(&lh[pi * g.nr + i0], lo);
                        atomicAdd(&lh[pi * g.nr + i0 + 1], up);
                    }
                }
            }
            head += n;
            cnt -= n;
        };
#pragma unroll 1
        for (int jc = 0; jc < PH_COLS; jc += FM_WAVE) {
            const Cand cj = colc[jc + lane];
            const int j = c0 + jc + lane;
#pragma unroll 1
            for (int k = 0; k < RW; ++k) {
                const int row = wid * RW + k;
                const int a = rowi[row];
                const bool keep = a >= 0 && j < natom && (sym ? j > a : true) && cand_pair<KIND>(rowc[row], cj, ct);
                const unsigned long long m = __ballot(keep);
                if (keep) q[(head + cnt + lanes_below(m)) & (2 * FM_WAVE - 1)] = (uint16_t)(row << 8 | (jc + lane));
                cnt += __popcll(m);
                if (cnt >= FM_WAVE) bin(FM_WAVE);
            }
        }
        if (cnt > 0) bin(cnt);
    }
    if (nshort) {
        for (int off = FM_WAVE / 2; off > 0; off >>= 1) shorts += __shfl_xor(shorts, off, FM_WAVE);
        if (lane == 0 && shorts) atomicAdd(&shorts_wg, shorts);
    }
    __syncthreads();
    for (int b = t; b < nb; b += NT) {
        const unsigned long long v = lh[b];
        if (v) atomicAdd(hist + b, v);
    }
    if (nshort && t == 0 && shorts_wg) atomicAdd(nshort, shorts_wg);
}

// d L / d pos for L = sum_p,i gbin[p][i] hist[p][i], every atom an absorber: pair (a, j) puts (1 - f, f) on the
// bins (i0, i0 + 1) of potential ipot[j]; its distance moves with pos_j - pos_a. A wavefront takes PG_ROWS atoms a,
// tests them against 64 atoms j at a time (float coordinates of PG_COLS atoms staged in LDS per workgroup), and
// evaluates each atom's queue of candidates 64 at a time; the lanes' sums are added in a fixed butterfly: no atomics,
// the same result on every run. Bound by VALU issue (82 % busy). 64 frames x 2000 atoms: 0.41 ms; one box of
// 4000: 0.074 ms (one thread per atom over all j in FP64: 1.15 ms, and 1.32 ms with its 16 workgroups on the chip).
constexpr int PG_WAVES = 4, PG_ROWS = 4, PG_COLS = 1024;

template <int KIND>
__global__ __launch_bounds__(FM_WAVE *PG_WAVES) void k_pair_grad(int natom, const double *pos, const int32_t *ipot,
                                                                 int npot, fm_pair_grid g, const double *gbin,
                                                                 double *grad) {
    __shared__ Cand colc[PG_COLS];
    __shared__ uint16_t queue[PG_WAVES][PG_ROWS][2 * FM_WAVE];
    const int c = blockIdx.y, t = threadIdx.x;
    const int wid = __builtin_amdgcn_readfirstlane(t / FM_WAVE), lane = t % FM_WAVE;
    const double *P = pos + (size_t)c * natom * 3;
    const double ref[3] = {P[0], P[1], P[2]};
    const CandTest ct = cand_test<KIND>(g);
    const int a0 = (blockIdx.x * PG_WAVES + wid) * PG_ROWS;
    Cand ca[PG_ROWS];
    double ga[PG_ROWS][3];
    int head[PG_ROWS], cnt[PG_ROWS];
#pragma unroll
    for (int k = 0; k < PG_ROWS; ++k) {
        ca[k] = cand_of<KIND>(P + 3 * (size_t)(a0 + k < natom ? a0 + k : 0), ref, g);
        ga[k][0] = ga[k][1] = ga[k][2] = 0.0;
        head[k] = cnt[k] = 0;
    }
    for (int c0 = 0; c0 < natom; c0 += PG_COLS) {
        __syncthreads();
        for (int j = t; j < PG_COLS; j += FM_WAVE * PG_WAVES)
            colc[j] = cand_of<KIND>(P + 3 * (size_t)(c0 + j < natom ? c0 + j : 0), ref, g);
        __syncthreads();
        // the first n queued candidates of atom a0 + k
        auto add = [&](int k, int n) {
            fm::wave_sync();
            if (lane < n) {
                const int a = a0 + k, j = c0 + queue[wid][k][(head[k] + lane) & (2 * FM_WAVE - 1)];
                const double pa[3] = {P[3 * (size_t)a], P[3 * (size_t)a + 1], P[3 * (size_t)a + 2]};
                double v[3], r;
                if (pair(pa, P + 3 * (size_t)j, g, v, r)) {
                    int i0;
                    double f, dfdr;
                    bin_of(r, g, i0, f, dfdr);
                    double dLdr = 0.0;
                    const int pj = ipot[j], pi = ipot[a];
                    if (pj >= 0 && pj < npot) {       // a the absorber, j the neighbor
                        const double *gb = gbin + (size_t)pj * g.nr + i0;
                        dLdr += (gb[1] - gb[0]) * dfdr;
                    }
                    if (pi >= 0 && pi < npot) {       // j the absorber, a the neighbor (same distance)
                        const double *gb = gbin + (size_t)pi * g.nr + i0;
                        dLdr += (gb[1] - gb[0]) * dfdr;
                    }
                    const double s = dLdr / r;        // d r / d pos_a = -(pos_j - pos_a) / r
#pragma unroll
                    for (int x = 0; x < 3; ++x) ga[k][x] -= s * v[x];
                }
            }
            head[k] += n;
            cnt[k] -= n;
        };
        const int c1 = natom - c0 < PG_COLS ? natom - c0 : PG_COLS;
#pragma unroll 1
        for (int jc = 0; jc < c1; jc += FM_WAVE) {
            const Cand cj = colc[jc + lane];
            const bool live = jc + lane < c1;
#pragma unroll
            for (int k = 0; k < PG_ROWS; ++k) {
                const bool keep = live && a0 + k < natom && cand_pair<KIND>(ca[k], cj, ct);
                const unsigned long long m = __ballot(keep);
                if (keep) queue[wid][k][(head[k] + cnt[k] + lanes_below(m)) & (2 * FM_WAVE - 1)] = (uint16_t)(jc + lane);
                cnt[k] += __popcll(m);
                if (cnt[k] >= FM_WAVE) add(k, FM_WAVE);
            }
        }
#pragma unroll
        for (int k = 0; k < PG_ROWS; ++k)       // the queue holds indices of this tile
            if (cnt[k] > 0) add(k, cnt[k]);
    }
#pragma unroll
    for (int k = 0; k < PG_ROWS; ++k) {
#pragma unroll
        for (int x = 0; x < 3; ++x)
            for (int off = FM_WAVE / 2; off > 0; off >>= 1) ga[k][x] += __shfl_xor(ga[k][x], off, FM_WAVE);
        if (lane < 3 && a0 + k < natom)
            grad[((size_t)c * natom + a0 + k) * 3 + lane] = lane == 0 ? ga[k][0] : lane == 1 ? ga[k][1] : ga[k][2];
    }
}

// ------------------------------------------------------------------------------------------------ table products
// chi[k] = sum_i hist[i] table[i][k] / div over the rows i of one potential's table: a workgroup sums TS_ROWS rows of
// 64 points (its wavefronts interleaved over the rows, their sums added in order) into part[chunk][k]; k_table_total
// adds the chunks of every potential in order. TT: the tables' type, HT: int64 fixed point (2^-32) or double.
// Reading the table once is the bound (5.7 MB per potential, 1.2 us at 4.7 TB/s); at 3.8 us it is mostly launch
// latency (the stacked FP64 copy of the tables, its transpose and library products it replaces took about 100 us).
// held: a copy of the table made on the way, or NULL (6.0 us with it; a copy of two tables by launches of their own added
// 18 us to a call).
constexpr int TS_ROWS = 128, TS_WAVES = 8;
template <class HT> __device__ __forceinline__ double hist_value(HT h) { return (double)h; }
template <> __device__ __forceinline__ double hist_value<long long>(long long h) { return (double)h * (1.0 / PH_ONE); }
template <class TT, class HT>
__global__ __launch_bounds__(FM_WAVE *TS_WAVES) void k_table_sum(int nr, int nk, const TT *table, const HT *hist,
                                                                 double *part, TT *held) {
    __shared__ double sm[TS_WAVES][FM_WAVE];
    const int w = threadIdx.x / FM_WAVE, lane = threadIdx.x % FM_WAVE;
    const int k = blockIdx.x * FM_WAVE + lane, i0 = blockIdx.y * TS_ROWS;
    TT x[TS_ROWS / TS_WAVES];
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < TS_ROWS / TS_WAVES; ++u) {
        const int i = i0 + u * TS_WAVES + w, ic = i < nr ? i : nr - 1;
        const double h = hist_value(hist[ic]);
        x[u] = table[(size_t)ic * nk + (k < nk ? k : nk - 1)];
        acc += i < nr ? h * (double)x[u] : 0.0;
    }
    if (held && k < nk) {
#pragma unroll
        for (int u = 0; u < TS_ROWS / TS_WAVES; ++u) {
            const int i = i0 + u * TS_WAVES + w;
            if (i < nr) held[(size_t)i * nk + k] = x[u];
        }
    }
    sm[w][lane] = acc;
    __syncthreads();
    if (w == 0 && k < nk) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < TS_WAVES; ++q) s += sm[q][lane];
        part[(size_t)blockIdx.y * nk + k] = s;
    }
}
__global__ __launch_bounds__(FM_WAVE * 4) void k_table_total(int nchunk, int nk, const double *part, double div,
                                                             double *chi) {
    const int k = blockIdx.x * FM_WAVE * 4 + threadIdx.x;
    if (k >= nk) return;
    double s = 0.0;
#pragma unroll 8
    for (int c = 0; c < nchunk; ++c) s += part[(size_t)c * nk + k];
    chi[k] = s / div;
}

// gbin[i] = sum_k table[i][k] g[k] / div: one wavefront per row.
template <class TT>
__global__ __launch_bounds__(FM_WAVE * 4) void k_table_grad(int nr, int nk, const TT *table, const double *g,
                                                            double div, double *gbin) {
    const int i = blockIdx.x * 4 + (int)(threadIdx.x / FM_WAVE), lane = threadIdx.x % FM_WAVE;
    if (i >= nr) return;
    double s = 0.0;
    for (int k = lane; k < nk; k += FM_WAVE) s += (double)table[(size_t)i * nk + k] * g[k];
    for (int off = FM_WAVE / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, FM_WAVE);
    if (lane == 0) gbin[i] = s / div;
}

const char *grid_problem(const fm_pair_grid *g) {
    if (!g) return "NULL grid";
    if (g->nr < 2) return "the distance grid needs nr >= 2";
    if (!(g->dr > 0.0)) return "dr must be positive";
    if (!(g->rmax > 0.0)) return "rmax must be positive";
    if (g->cell_kind < 0 || g->cell_kind > 2) return "cell_kind must be 0, 1 or 2";
    if (g->cell_kind == 1 && !(g->cell[0] > 0.0)) return "the cubic cell needs a positive length";
    return nullptr;
}

int launch_err(const char *what) {
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) return FM_OK;
    char buf[256];
    snprintf(buf, sizeof buf, "%s launch: %s", what, hipGetErrorString(e));
    return fm_set_err(FM_EHIP, buf);
}

}  // namespace

extern "C" {

int fm_pair_histogram(int32_t nconf, int32_t natom, const double *pos, int32_t nabs, const int32_t *absorbers,
                      const int32_t *ipot, int32_t npot, const fm_pair_grid *grid, int64_t *hist, int32_t *nshort,
                      void *stream) {
    const char *m = grid_problem(grid);
    if (m) return fm_set_err(FM_EINVAL, m);
    if (nconf < 0 || natom < 0 || npot < 1) return fm_set_err(FM_EINVAL, "fm_pair_histogram: bad sizes");
    const int na = absorbers ? nabs : natom;
    if (na < 0 || nconf > 65535) return fm_set_err(FM_EINVAL, "fm_pair_histogram: bad absorber count or more than 65535 configurations");
    if (nconf == 0 || natom == 0 || na == 0) return FM_OK;
    if (!pos || !ipot || !hist) return fm_set_err(FM_EINVAL, "fm_pair_histogram: NULL buffer");
    // every ordered pair adds one unit over two bins: nconf * na * (natom - 1) < 2^31 keeps every bin below overflow
    if ((double)nconf * na * (natom - 1) >= 2147483648.0)
        return fm_set_err(FM_EINVAL, "fm_pair_histogram: nconf * absorbers * (natom - 1) >= 2^31 pairs could overflow a "
                                     "bin; split the configurations over several calls");
    const size_t lds = sizeof(unsigned long long) * (size_t)npot * grid->nr;
    if (lds <= 144 * 1024) {   // the bins fit a workgroup's LDS
        const void *fn = grid->cell_kind == 0   ? (const void *)k_pair_hist_lds<0>
                         : grid->cell_kind == 1 ? (const void *)k_pair_hist_lds<1>
                                                : (const void *)k_pair_hist_lds<2>;
        if (lds > 48 * 1024) {
            hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return fm_set_err(FM_EHIP, hipGetErrorString(e));
        }
        int dev = 0, cus = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return fm_set_err(FM_EHIP, hipGetErrorString(e));
        const long items = (long)nconf * ((na + PH_ROWS - 1) / PH_ROWS) * ((natom + PH_COLS - 1) / PH_COLS);
        const long cap = cus > 0 ? cus : 1;
        const dim3 grd((unsigned)(items < cap ? items : cap)), blk(FM_WAVE * PH_WAVES);
        unsigned long long *const h = reinterpret_cast<unsigned long long *>(hist);
        hipStream_t st = (hipStream_t)stream;
        if (grid->cell_kind == 0)
            hipLaunchKernelGGL(k_pair_hist_lds<0>, grd, blk, lds, st, natom, nconf, pos, na, absorbers, ipot, npot, *grid, h, nshort);
        else if (grid->cell_kind == 1)
            hipLaunchKernelGGL(k_pair_hist_lds<1>, grd, blk, lds, st, natom, nconf, pos, na, absorbers, ipot, npot, *grid, h, nshort);
        else
            hipLaunchKernelGGL(k_pair_hist_lds<2>, grd, blk, lds, st, natom, nconf, pos, na, absorbers, ipot, npot, *grid, h, nshort);
    } else {
        hipLaunchKernelGGL(k_pair_hist, dim3((unsigned)na, (unsigned)nconf), dim3(PH_THREADS), 0, (hipStream_t)stream, natom,
                           pos, na, absorbers, ipot, npot, *grid, reinterpret_cast<unsigned long long *>(hist), nshort);
    }
    return launch_err("fm_pair_histogram");
}

int fm_pair_histogram_grad(int32_t nconf, int32_t natom, const double *pos, const int32_t *ipot, int32_t npot,
                           const fm_pair_grid *grid, const double *gbin, double *grad_pos, void *stream) {
    const char *m = grid_problem(grid);
    if (m) return fm_set_err(FM_EINVAL, m);
    if (nconf < 0 || natom < 0 || npot < 1 || nconf > 65535) return fm_set_err(FM_EINVAL, "fm_pair_histogram_grad: bad sizes");
    if (nconf == 0 || natom == 0) return FM_OK;
    if (!pos || !ipot || !gbin || !grad_pos) return fm_set_err(FM_EINVAL, "fm_pair_histogram_grad: NULL buffer");
    const int per = PG_WAVES * PG_ROWS;
    const dim3 grd((unsigned)((natom + per - 1) / per), (unsigned)nconf), blk(FM_WAVE * PG_WAVES);
    hipStream_t st = (hipStream_t)stream;
    if (grid->cell_kind == 0)
        hipLaunchKernelGGL(k_pair_grad<0>, grd, blk, 0, st, natom, pos, ipot, npot, *grid, gbin, grad_pos);
    else if (grid->cell_kind == 1)
        hipLaunchKernelGGL(k_pair_grad<1>, grd, blk, 0, st, natom, pos, ipot, npot, *grid, gbin, grad_pos);
    else
        hipLaunchKernelGGL(k_pair_grad<2>, grd, blk, 0, st, natom, pos, ipot, npot, *grid, gbin, grad_pos);
    return launch_err("fm_pair_histogram_grad");
}

size_t fm_pair_chi_workspace_bytes(int32_t npot, int32_t nr, int32_t nk) {
    if (npot < 1 || nr < 1 || nk < 1) return 0;
    return sizeof(double) * (size_t)npot * ((nr + TS_ROWS - 1) / TS_ROWS) * nk;
}

int fm_pair_chi(int32_t npot, const void *const *tables, const int32_t *rows, int32_t precision, int32_t nr, int32_t nk,
                const void *hist, int32_t fixed_point, double div, double *chi, void *workspace, size_t workspace_bytes,
                void *stream) {
    return fm_pair_chi_held(npot, tables, rows, precision, nr, nk, hist, fixed_point, div, chi, nullptr, workspace,
                            workspace_bytes, stream);
}

int fm_pair_chi_held(int32_t npot, const void *const *tables, const int32_t *rows, int32_t precision, int32_t nr,
                     int32_t nk, const void *hist, int32_t fixed_point, double div, double *chi, void *held,
                     void *workspace, size_t workspace_bytes, void *stream) {
    if (npot < 1 || nr < 1 || nk < 1) return fm_set_err(FM_EINVAL, "fm_pair_chi: bad sizes");
    if (precision != 32 && precision != 64) return fm_set_err(FM_EINVAL, "precision must be 32 or 64");
    if (!tables || !rows || !hist || !chi || !workspace) return fm_set_err(FM_EINVAL, "fm_pair_chi: NULL buffer");
    if (workspace_bytes < fm_pair_chi_workspace_bytes(npot, nr, nk))
        return fm_set_err(FM_EINVAL, "fm_pair_chi: workspace smaller than fm_pair_chi_workspace_bytes");
    const int chunks = (nr + TS_ROWS - 1) / TS_ROWS;
    const dim3 grd((unsigned)((nk + FM_WAVE - 1) / FM_WAVE), (unsigned)chunks), blk(FM_WAVE * TS_WAVES);
    hipStream_t st = (hipStream_t)stream;
    double *part = (double *)workspace;
    for (int p = 0; p < npot; ++p) {
        if (!tables[p] || rows[p] < 0) return fm_set_err(FM_EINVAL, "fm_pair_chi: NULL table or negative row");
        double *const out = part + (size_t)p * chunks * nk;
        const size_t at = (size_t)p * nr * nk;
        float *const h32 = held ? (float *)held + at : nullptr;
        double *const h64 = held ? (double *)held + at : nullptr;
        if (fixed_point) {
            const long long *h = (const long long *)hist + (size_t)rows[p] * nr;
            if (precision == 32)
                hipLaunchKernelGGL((k_table_sum<float, long long>), grd, blk, 0, st, nr, nk, (const float *)tables[p], h,
                                   out, h32);
            else
                hipLaunchKernelGGL((k_table_sum<double, long long>), grd, blk, 0, st, nr, nk, (const double *)tables[p],
                                   h, out, h64);
        } else {
            const double *h = (const double *)hist + (size_t)rows[p] * nr;
            if (precision == 32)
                hipLaunchKernelGGL((k_table_sum<float, double>), grd, blk, 0, st, nr, nk, (const float *)tables[p], h,
                                   out, h32);
            else
                hipLaunchKernelGGL((k_table_sum<double, double>), grd, blk, 0, st, nr, nk, (const double *)tables[p],
                                   h, out, h64);
        }
    }
    hipLaunchKernelGGL(k_table_total, dim3((unsigned)((nk + FM_WAVE * 4 - 1) / (FM_WAVE * 4))), dim3(FM_WAVE * 4), 0, st,
                       npot * chunks, nk, part, div, chi);
    return launch_err("fm_pair_chi");
}

int fm_pair_chi_grad(int32_t npot, const void *const *tables, const int32_t *rows, int32_t precision, int32_t nr,
                     int32_t nk, const double *gchi, double div, double *gbin, void *stream) {
    if (npot < 1 || nr < 1 || nk < 1) return fm_set_err(FM_EINVAL, "fm_pair_chi_grad: bad sizes");
    if (precision != 32 && precision != 64) return fm_set_err(FM_EINVAL, "precision must be 32 or 64");
    if (!tables || !rows || !gchi || !gbin) return fm_set_err(FM_EINVAL, "fm_pair_chi_grad: NULL buffer");
    hipStream_t st = (hipStream_t)stream;
    for (int p = 0; p < npot; ++p) {
        if (!tables[p] || rows[p] < 0) return fm_set_err(FM_EINVAL, "fm_pair_chi_grad: NULL table or negative row");
        const dim3 grd((unsigned)((nr + 3) / 4)), blk(FM_WAVE * 4);
        double *const out = gbin + (size_t)rows[p] * nr;
        if (precision == 32)
            hipLaunchKernelGGL(k_table_grad<float>, grd, blk, 0, st, nr, nk, (const float *)tables[p], gchi, div, out);
        else
            hipLaunchKernelGGL(k_table_grad<double>, grd, blk, 0, st, nr, nk, (const double *)tables[p], gchi, div, out);
    }
    return launch_err("fm_pair_chi_grad");
}

}  // extern "C"
