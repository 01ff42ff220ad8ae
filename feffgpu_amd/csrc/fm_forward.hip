// Fused path-stage forward kernels for gfx950 and the C ABI that launches them.
//
// A workgroup of 4 wavefronts holds G paths (1, 2, 4 or 8: as many as fit the LDS) of the same edge and leg count.
// Per path one wavefront computes the leg geometry in FP64 (one lane per leg) and the rotation tables
// d^l_{m1 m2}(beta_s) of every leg into LDS (one lane per (leg, pair)). The (path, energy) pairs are then cut into
// energy bands of the edge's plan: a wavefront runs whole bands, lane (path j, energy i) = j * (64 / G) + i, so its
// lanes loop over similar numbers of partial waves, and the bands are spread over the wavefronts so that their
// loads balance. Every lane evaluates the Rehr-Albers amplitude at its energy: the termination matrix T, then the
// scattering matrices F_{n-1} ... F_1 multiplied into U = T F_{n-1} ... F_s, each F streamed over the lane's partial
// waves with the spherical-wave recursion of its two legs kept in registers; cchi = tr(U) cfac. The fine grid
// (amplitude and unwrapped phase interpolated to q, chi = A sin(Phi + 2 q reff)) is one wavefront's epilogue per
// path.
//
// Reference semantics: GPUPathStage.cchi / chi_fine (src/feffgpu/stage.py:235-388), the literal port
// genfmt.PathStage (src/feffgpu/genfmt.py:395-445) and the path-list gather/sum of
// src/feffgpu/exafs/forward.py:143-163.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <type_traits>

#include "fm_device.h"
#include "fm_internal.h"
#include "fm_path.h"

using namespace fm;

thread_local char g_err[512] = "";
int fm_set_err(int code, const char *msg) {
    snprintf(g_err, sizeof g_err, "%s", msg);
    return code;
}

// LDS a workgroup may take when the paths per workgroup are chosen (bytes): FP32 forward, FP32 adjoint, FP64
// forward, FP64 adjoint.
static std::atomic<size_t> g_lds_budget[4] = {{80 * 1024}, {160 * 1024}, {160 * 1024}, {160 * 1024}};
size_t fm_lds_budget(int kernel) { return g_lds_budget[kernel & 3].load(std::memory_order_relaxed); }

namespace {

struct KArgs {
    fm_edge ed;           // the edge of every path of this launch
    fm_bands bp;          // its band plan for gp paths per workgroup
    int gp;
    int npath_bucket;     // paths in this launch
    int first;            // offset into order[]
    const int32_t *order;
    PathSrc src;
    void *cchi_out;       // mode 0
    fm_grid G;            // mode 1
    void *chi_path;
    double *reff_out;
    int edge_id;          // index of the edge (rows of the grid's jq / fq)
    int nleg;             // the leg count of every path of this launch
    size_t path_bytes;    // LDS per path of a workgroup
    unsigned *tickets;    // the path groups' counter pair of a persistent launch, or NULL (fixed assignment)
    void *keep;           // the bucket's kept scattering matrices (written), or NULL
    uint32_t *rows;       // split launch: the output rows, path p's at rows + p row_words
    size_t row_words;
};

int set_err(int code, const char *msg) {
    snprintf(g_err, sizeof g_err, "%s", msg);
    return code;
}
int hip_err(hipError_t e, const char *where) {
    snprintf(g_err, sizeof g_err, "%s: %s", where, hipGetErrorString(e));
    return FM_EHIP;
}


// ---- The split launch. The geometry of a path and its fine grid are chains of FP64 latencies with little parallelism,
// which k_forward's two wavefronts per SIMD hide badly: of 1220 us (77 005 paths of 3 legs, K edge, FP32) they were 350
// and 180. So k_rows fills a record per path (16 lanes each, seven wavefronts per SIMD) in the path's own row of the
// output, k_forward reads the record and leaves cchi there, and k_fine turns it into chi(k): 904 us together (L3 edge,
// 51 213 paths of 3 legs: 1137 -> 765; single scattering, 32 828 paths: 244 -> 209; FP64, 12 838 paths of 3 legs: 468 ->
// 326). Below SPLIT_MIN paths the two more launches cost more than that (700 paths of 3 legs 42 against 44 us, 1290 paths
// 66 against 56).
// A record: the leg lengths, cos/sin of eta and 2 eta, of beta and beta/2 (9 n doubles), R, reff, prod r, ok and the
// potentials; after the bands the row holds cchi (2 E of T), reff (A) and ok. 32-bit words: rows need not be 8-byte
// aligned.
constexpr int SPLIT_MIN = 1280;
constexpr int SPLIT_PATHS = 1 << 25;     // of one launch of k_rows or k_fine, whose threads must stay below 2^32
__host__ __device__ constexpr int rec_words(int n) { return 2 * (9 * n + 3) + n + 1; }
__device__ __forceinline__ void put_double(uint32_t *w, double v) { __builtin_memcpy(w, &v, 8); }
__device__ __forceinline__ double get_double(const uint32_t *w) {
    uint32_t x[2] = {w[0], w[1]};
    double v;
    __builtin_memcpy(&v, x, 8);
    return v;
}
__global__ __launch_bounds__(256) void k_rows(KArgs a) {
    __shared__ PathLDS gs[16];
    const int t = threadIdx.x, n = a.nleg, lane = t & 15;
    const int q = blockIdx.x * 16 + t / 16;
    const int s0 = q < a.npath_bucket ? q : blockIdx.x * 16;
    const int p = a.order ? a.order[a.first + s0] : a.first + s0;
    PathLDS &g = gs[t / 16];
    int ei;
    load_path_group(a.src, p, g, ei, n, lane, true);
    if (q >= a.npath_bucket) return;
    uint32_t *const w = a.rows + (size_t)p * a.row_words;
    if (lane < n) {
        const int J = lane + 1;
        const double v[9] = {g.r[J], g.c1[J], g.s1[J], g.c2[J], g.s2[J], g.cb[J], g.sb[J], g.ch[J], g.sh[J]};
#pragma unroll
        for (int f = 0; f < 9; ++f) put_double(w + 2 * (f * n + lane), v[f]);
        w[2 * (9 * n + 3) + 1 + lane] = (uint32_t)g.ipot[lane];
    }
    if (lane == 0) {
        put_double(w + 2 * (9 * n), g.R);
        put_double(w + 2 * (9 * n + 1), g.reff);
        put_double(w + 2 * (9 * n + 2), g.prod_r);
        w[2 * (9 * n + 3)] = (uint32_t)g.ok;
    }
}
// The records of the wavefront's paths j = wid, wid + 4, ... < G of group blk (np <= 2) into LDS, their numbers into
// pidx and pval: every lane fetches its own path's number and item, so that both latencies are waited for once.
__device__ __forceinline__ void load_records(const KArgs &a, int blk, int G, int wid, int lane, unsigned char *smem, int *pidx,
                                             int *pval) {
    const int n = a.nleg, np = wid < G ? (G - 1 - wid) / 4 + 1 : 0;
    auto path = [&](int j, bool &valid) {
        const int slot = blk * G + j;
        valid = slot < a.npath_bucket;
        const int s0 = valid ? slot : blk * G;
        return a.order ? a.order[a.first + s0] : a.first + s0;
    };
    // R, reff, prod r; ok and the potentials
    const int q = lane / (n + 4), k = lane - q * (n + 4), j = wid + 4 * (q < np ? q : 0);
    bool valid;
    const int p = path(j < G ? j : 0, valid);
    const uint32_t *const w = a.rows + (size_t)p * a.row_words + 2 * 9 * n;
    double d = 0.0;
    uint32_t v = 0;
    if (k < 3) d = get_double(w + 2 * k); else v = w[6 + k - 3];
    for (int x = lane; x < np * 9 * n; x += FM_WAVE) {
        const int xq = x / (9 * n), i = x - xq * 9 * n, f = i / n, J = i - f * n + 1, xj = wid + 4 * xq;
        bool xv;
        const double t = get_double(a.rows + (size_t)path(xj, xv) * a.row_words + 2 * i);
        PathLDS &g = *reinterpret_cast<PathLDS *>(smem + (size_t)xj * a.path_bytes);
        double *const to = f == 0 ? g.r : f < 5 ? g.c1 + (f - 1) * (FM_MAX_LEGS + 1) : g.cb + (f - 5) * (FM_MAX_LEGS + 1);
        to[J] = t;
    }
    if (q < np) {
        PathLDS &g = *reinterpret_cast<PathLDS *>(smem + (size_t)j * a.path_bytes);
        if (k == 0) {
            g.R = d;
            g.n = n;
            pidx[j] = p;
            pval[j] = valid ? 1 : 0;
        } else if (k == 1) {
            g.reff = d;
        } else if (k == 2) {
            g.prod_r = d;
        } else if (k == 3) {
            g.ok = (int)v;
        } else {
            g.ipot[k - 4] = (int)v;
            if (k == 4) g.ipot[n] = (int)v;
        }
    }
}
// The fine grid of the paths whose rows hold cchi, one wavefront per path.
template <class T> __global__ __launch_bounds__(FM_WAVE * 4) void k_fine(KArgs a, size_t wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wid = threadIdx.x / FM_WAVE, lane = lane_id(), s0 = blockIdx.x * 4 + wid;
    if (s0 >= a.npath_bucket) return;
    const int p = a.order ? a.order[a.first + s0] : a.first + s0, E = a.ed.E, nk = a.G.nk;
    T *const amp = reinterpret_cast<T *>(smem + (size_t)wid * wave_bytes);
    double *const ang = reinterpret_cast<double *>(smem + (size_t)wid * wave_bytes + align16(sizeof(T) * (size_t)E));
    uint32_t *const w = a.rows + (size_t)p * a.row_words;
    T *const out = reinterpret_cast<T *>(w);
    const uint32_t *const meta = w + 2 * E * (sizeof(T) / 4);
    const double reff_A = get_double(meta);
    if (meta[2]) {
        for (int e = lane; e < E; e += FM_WAVE) {
            const cx<T> c = mk<T>(out[2 * e], out[2 * e + 1]);
            amp[e] = (T)sqrt((double)c.r * c.r + (double)c.i * c.i + 1e-30);
            ang[e] = (double)atan2(c.i, c.r);
        }
        wave_sync();
        fine_grid<T>(a.ed, a.G.jq + (size_t)a.edge_id * nk, a.G.fq + (size_t)a.edge_id * nk, a.G.q, nk, reff_A,
                     a.src.P.sigma2 ? a.src.P.sigma2[p] : 0.0, amp, ang, out,
                     a.G.S ? a.G.S + (size_t)a.edge_id * nk * a.G.sstride : nullptr, a.G.sstride);
    } else {
        for (int i = lane; i < nk; i += FM_WAVE) out[i] = (T)__builtin_nan("");
    }
}

// SPLIT: of a split launch (the records of multiple-scattering paths read, cchi left in the rows of mode 1).
template <class T, int SET, bool SPLIT = false>
__global__ __launch_bounds__(FM_WAVE * 4) __attribute__((amdgpu_waves_per_eu(FM_WPE(T)))) void k_forward(KArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int pidx[8], pval[8], tslot;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FM_WAVE);
    const int lane = lane_id();
    const fm_edge &ed = a.ed;
    const int G = a.gp, cap = FM_WAVE / G;
    const int ltab = ed.L1 + 1, E = ed.E;
    const int nl = a.nleg;
    const size_t off_W = align16(sizeof(PathLDS));
    const size_t off_amp = off_W + (SET < FM_SET_SS ? align16(sizeof(T) * rot_elems(nl, ltab)) : 0);
    const size_t off_ang = off_amp + align16(sizeof(T) * (size_t)E);
    const int jl = lane / cap, il = lane % cap;      // this lane's path and energy within a band
    unsigned char *lbase = smem + (size_t)jl * a.path_bytes;
    const PathLDS &gl = *reinterpret_cast<const PathLDS *>(lbase);
    const T *Wl = reinterpret_cast<const T *>(lbase + off_W);
    for (int blk = first_group(a.tickets, tslot); blk * G < a.npath_bucket; blk = next_group(a.tickets, tslot, blk)) {
        // ---- setup. Single scattering (no tables): the wavefront's paths j = wid, wid + 4 at once, a 16-lane group
        // each (G <= 8); multiple scattering: one path after the other (measured faster there, the two workgroups of
        // a CU overlapping their setups)
        if constexpr (SET >= FM_SET_SS) {
            const int j = wid + 4 * (lane >> 4);
            const bool act = j < G;
            const int slot = blk * G + j;
            const bool valid = act && slot < a.npath_bucket;
            const int s0 = valid ? slot : blk * G;
            const int p = a.order ? a.order[a.first + s0] : a.first + s0;
            PathLDS &g = *reinterpret_cast<PathLDS *>(smem + (size_t)(act ? j : 0) * a.path_bytes);
            int ei;
            load_path_group(a.src, p, g, ei, nl, lane & 15, act, false);   // single scattering: no tables
            if (act && (lane & 15) == 0) { pidx[j] = p; pval[j] = valid ? 1 : 0; }
        } else if constexpr (SPLIT) {
            load_records(a, blk, G, wid, lane, smem, pidx, pval);
            wave_sync();
        } else {
            for (int j = wid; j < G; j += 4) {
                const int slot = blk * G + j;
                const bool valid = slot < a.npath_bucket;
                const int s0 = valid ? slot : blk * G;
                const int p = a.order ? a.order[a.first + s0] : a.first + s0;
                PathLDS &g = *reinterpret_cast<PathLDS *>(smem + (size_t)j * a.path_bytes);
                int ei;
                load_path(a.src, p, g, ei, nl);
                if (lane == 0) { pidx[j] = p; pval[j] = valid ? 1 : 0; }
            }
        }
        // the tables' coefficients 8 rows at a time in a split launch (which keeps matrices 6% faster than row by row; the
        // unsplit kernel, short of registers, is faster row by row)
        if constexpr (SET < FM_SET_SS)
            build_tables<T, SET, false, SPLIT ? 8 : 1>(ed, smem, a.path_bytes, off_W, 0, wid, 4, G, nl, ltab);
        __syncthreads();
        // ---- energies: the bands of this wavefront, each wavefront stepping from one of its bands to the next
        auto next_band = [&](int b) {
            for (++b; b < a.bp.nband && a.bp.wave[b] != wid; ++b) {}
            return b;
        };
        for (int b = next_band(-1); b < a.bp.nband; b = next_band(b)) {
            const int e0 = a.bp.start[b], nb = a.bp.start[b + 1] - e0;
            const bool active = il < nb && pval[jl];
            const int e = e0 + (il < nb ? il : nb - 1);
            cx<T> c;
            if constexpr (SET >= FM_SET_SS) {
                c = ss_cchi<T, SET - FM_SET_SS + 1>(ed, gl, e);
            } else {
                // this lane's (path, energy) in the kept rows, written by active lanes only
                T *kp = (a.keep && active)
                            ? reinterpret_cast<T *>(a.keep) + ((size_t)(blk * G + jl) * keep_rows<SET>(nl) * E + e) * 2
                            : nullptr;
                c = path_cchi<T, SET>(ed, gl, Wl, ltab, e, nl, kp);
            }
            if (active) {
                if (a.src.mode == 0) {
                    T *o = reinterpret_cast<T *>(a.cchi_out) + ((size_t)pidx[jl] * E + e) * 2;
                    o[0] = gl.ok ? c.r : (T)__builtin_nan("");
                    o[1] = gl.ok ? c.i : (T)__builtin_nan("");
                } else if constexpr (SPLIT) {
                    T *const o = reinterpret_cast<T *>(a.rows + (size_t)pidx[jl] * a.row_words);
                    o[2 * e] = c.r;
                    o[2 * e + 1] = c.i;
                } else {
                    T *amp = reinterpret_cast<T *>(lbase + off_amp);
                    double *ang = reinterpret_cast<double *>(lbase + off_ang);
                    amp[e] = (T)sqrt((double)c.r * c.r + (double)c.i * c.i + 1e-30);
                    ang[e] = (double)atan2(c.i, c.r);
                }
            }
        }
        __syncthreads();
        // ---- epilogue: one wavefront per path
        for (int j = wid; j < G; j += 4) {
            if (!pval[j]) continue;
            unsigned char *base = smem + (size_t)j * a.path_bytes;
            const PathLDS &g = *reinterpret_cast<const PathLDS *>(base);
            const int p = pidx[j];
            const double reff_A = g.ok ? g.reff * FM_BOHR : __builtin_nan("");
            if (lane == 0 && a.reff_out) a.reff_out[p] = reff_A;
            if constexpr (SPLIT) {
                if (a.src.mode == 1 && lane == 0) {
                    uint32_t *const w = a.rows + (size_t)p * a.row_words + 2 * E * (sizeof(T) / 4);
                    put_double(w, reff_A);
                    w[2] = (uint32_t)g.ok;
                }
            } else if (a.src.mode == 1) {
                const int nk = a.G.nk;
                T *out = reinterpret_cast<T *>(a.chi_path) + (size_t)p * nk;
                if (g.ok)
                    fine_grid<T>(ed, a.G.jq + (size_t)a.edge_id * nk, a.G.fq + (size_t)a.edge_id * nk, a.G.q, nk, reff_A,
                                 a.src.P.sigma2 ? a.src.P.sigma2[p] : 0.0, reinterpret_cast<T *>(base + off_amp),
                                 reinterpret_cast<double *>(base + off_ang), out,
                                 a.G.S ? a.G.S + (size_t)a.edge_id * nk * a.G.sstride : nullptr, a.G.sstride);
                else
                    for (int i = lane; i < nk; i += FM_WAVE) out[i] = (T)__builtin_nan("");
            }
        }
        __syncthreads();
    }
    release_groups(a.tickets);
}

// The scattering matrices alone, in the kept rows' layout (for an adjoint whose forward kept none): k_forward's setup
// and bands without the termination and the chain.
template <class T, int SET>
__global__ __launch_bounds__(FM_WAVE * 4) __attribute__((amdgpu_waves_per_eu(FM_WPE(T)))) void k_matrices(KArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int L = lamdef(SET).L, L0 = lamdef(SET).L0;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FM_WAVE);
    const int lane = lane_id();
    const fm_edge &ed = a.ed;
    const int G = a.gp, cap = FM_WAVE / G;
    const int ltab = ed.L1 + 1, E = ed.E, n = a.nleg, blk = blockIdx.x;
    const size_t off_W = align16(sizeof(PathLDS));
    const int jl = lane / cap, il = lane % cap;      // this lane's path and energy within a band
    unsigned char *lbase = smem + (size_t)jl * a.path_bytes;
    const PathLDS &g = *reinterpret_cast<const PathLDS *>(lbase);
    const T *W = reinterpret_cast<const T *>(lbase + off_W);
    for (int j = wid; j < G; j += 4) {
        const int slot = blk * G + j;
        const int s0 = slot < a.npath_bucket ? slot : blk * G;
        int ei;
        load_path(a.src, a.order ? a.order[a.first + s0] : a.first + s0,
                  *reinterpret_cast<PathLDS *>(smem + (size_t)j * a.path_bytes), ei, n);
    }
    build_tables<T, SET, false, 1>(ed, smem, a.path_bytes, off_W, 0, wid, 4, G, n, ltab);
    __syncthreads();
    const int tlstride = 2 * E;
    const bool valid = blk * G + jl < a.npath_bucket;
    for (int b = 0; b < a.bp.nband; ++b) {
        if (a.bp.wave[b] != wid) continue;
        const int e0 = a.bp.start[b], nb = a.bp.start[b + 1] - e0;
        const bool active = il < nb && valid;
        const int e = e0 + (il < nb ? il : nb - 1);
        T *kp = reinterpret_cast<T *>(a.keep) + ((size_t)(blk * G + (valid ? jl : 0)) * keep_rows<SET>(n) * E + e) * 2;
        const cx<T> ck = mk<T>((T)ed.ck[2 * e], (T)ed.ck[2 * e + 1]);
        auto block = [&](int s, auto nr, auto nc) {
            constexpr int NR = decltype(nr)::value, NC = decltype(nc)::value;
            const int ip = g.ipot[s];
            const T *tl = TL<T>::tl(ed) + ((size_t)ip * ltab) * tlstride + 2 * e;
            cx<T> Ft[FM_NREP];
            fblock<T, SET, NR, NC, true>(Ft, ck, (T)g.r[s + 1], (T)g.r[s], ed.lmax[(size_t)ip * E + e] + 1,
                                         W + (size_t)(s - 1) * ltab * FM_NREP, tl, tlstride);
            if (active) keep_store<T, SET, NR, NC>(kp + (size_t)2 * E * keep_off<SET>(n, s), E, Ft);
        };
        block(1, std::integral_constant<int, L>{}, std::integral_constant<int, L0>{});
#pragma unroll 1
        for (int s = 2; s < n - 1; ++s) block(s, std::integral_constant<int, L>{}, std::integral_constant<int, L>{});
        block(n - 1, std::integral_constant<int, L0>{}, std::integral_constant<int, L>{});
    }
}

// GPUPathStage.chi_fine on its own: one wave per path reads cchi [npath][E] and runs the fine-grid epilogue.
template <class T>
__global__ __launch_bounds__(FM_WAVE *WPB_MAX) void k_chi_fine(fm_edge ed, int npath, const T *cchi, const double *reff,
                                                                fm_grid G, T *chi, size_t wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wid = threadIdx.x / FM_WAVE, lane = lane_id();
    const int wpb = blockDim.x / FM_WAVE;
    unsigned char *base = smem + (size_t)wid * wave_bytes;
    T *amp = reinterpret_cast<T *>(base);
    double *ang = reinterpret_cast<double *>(base + align16(sizeof(T) * (size_t)ed.E));
    for (int p = blockIdx.x * wpb + wid; p < npath; p += gridDim.x * wpb) {
        for (int e = lane; e < ed.E; e += FM_WAVE) {
            const T cr = cchi[((size_t)p * ed.E + e) * 2], ci = cchi[((size_t)p * ed.E + e) * 2 + 1];
            amp[e] = (T)sqrt((double)cr * cr + (double)ci * ci + 1e-30);
            ang[e] = (double)atan2(ci, cr);
        }
        wave_sync();
        fine_grid<T>(ed, G.jq, G.fq, G.q, G.nk, reff[p], 0.0, amp, ang, chi + (size_t)p * G.nk);
        wave_sync();
    }
}

// The same with a dense interpolation matrix S [nk][sstride]: a contraction of S with the amplitudes and phases of 64
// paths per workgroup, lanes over the paths, DR rows of S per wavefront. S is wave-uniform (scalar loads, an operand of
// the FP64 multiply-adds), the amplitudes and phases come from LDS, DE energies at a time, and are read once per DR
// rows; the sums run over the energies in order, as in fine_grid. Bound by the latency of the scalar loads and of the
// amplitudes (few wavefronts: DR = 4). One wavefront per path with the lanes over the rows (k_chi_fine) reads all of S
// per path, a cache line per lane and energy: 2048 paths, E = 59, nk = 361, FP32: 96 us, here 19 us (DR = 8: 25).
constexpr int DR = 4, DW = 8, DE = 64, DLD = FM_WAVE + 1;
typedef const __attribute__((address_space(4))) double *scalar_ptr;
template <class T>
__global__ __launch_bounds__(FM_WAVE *DW) void k_chi_dense(fm_edge ed, int npath, const T *cchi, const double *reff,
                                                           fm_grid G, T *chi) {
    __shared__ T amp[DE * DLD];
    __shared__ double ang[DE * DLD], tot[DW][FM_WAVE];
    static_assert(DE == 8 * DW, "8 energies per wavefront");
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FM_WAVE), lane = lane_id();
    const int E = ed.E, p0 = blockIdx.x * FM_WAVE, np = npath - p0 < FM_WAVE ? npath - p0 : FM_WAVE;
    const int i0 = (blockIdx.y * DW + wid) * DR;
    double sa[DR], sp[DR];
    scalar_ptr Sr[DR];
#pragma unroll
    for (int r = 0; r < DR; ++r) {
        sa[r] = sp[r] = 0.0;
        const int i = i0 + r < G.nk ? i0 + r : G.nk - 1;
        Sr[r] = (scalar_ptr)(uintptr_t)(G.S + (size_t)i * G.sstride);
    }
    const int j = lane < np ? lane : np - 1;
    const T *const c0 = cchi + (size_t)(p0 + j) * E * 2;
    double carry = 0.0;
    for (int e0 = 0; e0 < E; e0 += DE) {
        const int ne = E - e0 < DE ? E - e0 : DE;
        // energies e0 + 8 wid .. + 7 of path `lane`: amplitudes, and the phase steps wrapped to (-pi, pi], summed over
        // the thread's 8 and then over the wavefronts
        double d[8], last = 0.0;
        {
            const int eb = e0 + wid * 8;
            const T *cp = c0 + 2 * (size_t)(eb > 0 ? (eb <= E ? eb - 1 : E - 1) : 0);
            last = eb > 0 ? (double)atan2(cp[1], cp[0]) : 0.0;
            double s = 0.0;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = eb + u < E ? eb + u : E - 1;
                const T cr = c0[2 * (size_t)e], ci = c0[2 * (size_t)e + 1];
                amp[(wid * 8 + u) * DLD + lane] = (T)sqrt((double)cr * cr + (double)ci * ci + 1e-30);
                const double a = (double)atan2(ci, cr), x = a - last;
                s += eb + u == 0 ? a : eb + u < E ? x - FM_TWO_PI * rint(x / FM_TWO_PI) : 0.0;
                d[u] = s;
                last = a;
            }
            tot[wid][lane] = s;
        }
        __syncthreads();
        double before = carry;
#pragma unroll
        for (int w = 0; w < DW; ++w) {
            if (w < wid) before += tot[w][lane];
            carry += tot[w][lane];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) ang[(wid * 8 + u) * DLD + lane] = before + d[u];
        __syncthreads();
        if (i0 < G.nk) {
#pragma unroll 4
            for (int e = 0; e < ne; ++e) {
                const double av = (double)amp[e * DLD + lane], pv = ang[e * DLD + lane];
#pragma unroll
                for (int r = 0; r < DR; ++r) {
                    const double s = Sr[r][e0 + e];
                    sa[r] += s * av;
                    sp[r] += s * pv;
                }
            }
        }
        __syncthreads();
    }
    if (lane >= np) return;
    const double R = reff[p0 + lane];
#pragma unroll
    for (int r = 0; r < DR; ++r) {
        const int i = i0 + r;
        if (i >= G.nk) break;
        double ph = sp[r] + 2.0 * G.q[i] * R;
        ph -= FM_TWO_PI * rint(ph / FM_TWO_PI);
        T v;
        if constexpr (sizeof(T) == 4) v = (T)sa[r] * sinf((float)ph);
        else v = (T)sa[r] * sin(ph);
        chi[(size_t)(p0 + lane) * G.nk + i] = v;
    }
}

// ------------------------------------------------------------------------------------------------ launch helpers
int set_for(const fm_edge &ed, int nleg) {
    if (nleg == 2) return FM_SET_SS + ed.ilinit - 1;
    return ed.ilinit <= 1 ? 0 : 1;
}

// Paths per workgroup: the policy's, else the largest plan within the LDS budget (by default room for two workgroups
// per CU), else the largest that fits one workgroup. Grid: one workgroup per group, or the policy's persistent grid.
template <class T, int SET, bool SPLIT> hipError_t launch_main(KArgs &a, const fm_launch &pol, hipStream_t st) {
    const fm_edge &ed = a.ed;
    a.path_bytes = path_stride(align16(sizeof(PathLDS)) +
                               (SET < FM_SET_SS ? align16(sizeof(T) * rot_elems(a.nleg, ed.L1 + 1)) : 0) +
                               align16(sizeof(T) * ed.E) + align16(sizeof(double) * ed.E));
    const int g = choose_gpaths(ed, a.path_bytes, fm_lds_budget(sizeof(T) == 4 ? 0 : 2), pol.gpaths,
                                a.npath_bucket, FM_WPE(T));
    if (g == -2) return hipErrorInvalidConfiguration;
    if (g < 0) return hipErrorInvalidValue;
    a.gp = 1 << g;
    a.bp = ed.bands[g];
    const size_t shm = a.path_bytes * a.gp;
    const void *fn = (const void *)k_forward<T, SET, SPLIT>;
    if (shm > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) return e;
    }
    long blocks = 0;
    hipError_t e = launch_grid(fn, shm, (a.npath_bucket + a.gp - 1) / a.gp, pol.grid, &blocks);
    if (e != hipSuccess) return e;
    if (blocks == 0) return hipSuccess;
    a.tickets = pol.grid != 0 ? pol.tickets : nullptr;
    const auto pieces = [&](auto run) {
        for (long f = 0; f < a.npath_bucket; f += SPLIT_PATHS) {
            KArgs b = a;
            b.first = a.first + (int)f;
            b.npath_bucket = a.npath_bucket - f < SPLIT_PATHS ? (int)(a.npath_bucket - f) : SPLIT_PATHS;
            run(b);
        }
    };
    if (SPLIT && SET < FM_SET_SS)
        pieces([&](const KArgs &b) {
            hipLaunchKernelGGL(k_rows, dim3((unsigned)((b.npath_bucket + 15) / 16)), dim3(256), 0, st, b);
        });
    hipLaunchKernelGGL((k_forward<T, SET, SPLIT>), dim3((unsigned)blocks), dim3(FM_WAVE * 4), shm, st, a);
    if (SPLIT && a.src.mode == 1) {
        const size_t wb = align16(sizeof(T) * (size_t)ed.E) + align16(sizeof(double) * (size_t)ed.E);
        pieces([&](const KArgs &b) {
            hipLaunchKernelGGL(k_fine<T>, dim3((unsigned)((b.npath_bucket + 3) / 4)), dim3(FM_WAVE * 4), 4 * wb, st, b, wb);
        });
    }
    return hipGetLastError();
}

template <class T, int SET> hipError_t launch_forward(KArgs &a, const fm_launch &pol, hipStream_t st) {
    // the split launch, where the output rows hold what it leaves there
    const size_t cw = 2 * (size_t)a.ed.E * (sizeof(T) / 4);      // words of a path's cchi
    a.rows = reinterpret_cast<uint32_t *>(a.src.mode == 1 ? a.chi_path : a.cchi_out);
    a.row_words = a.src.mode == 1 ? (size_t)a.G.nk * (sizeof(T) / 4) : cw;
    const size_t need = SET < FM_SET_SS ? (size_t)rec_words(a.nleg) : 0;
    const bool fits = a.row_words >= need && (a.src.mode == 0 ? SET < FM_SET_SS : a.row_words >= cw + 3);
    if (a.npath_bucket > SPLIT_MIN && fits) return launch_main<T, SET, true>(a, pol, st);
    return launch_main<T, SET, false>(a, pol, st);
}

template <class T, int SET> hipError_t launch_matrices(KArgs &a, const fm_launch &pol, hipStream_t st) {
    const fm_edge &ed = a.ed;
    a.path_bytes = path_stride(align16(sizeof(PathLDS)) + align16(sizeof(T) * rot_elems(a.nleg, ed.L1 + 1)));
    const int g = choose_gpaths(ed, a.path_bytes, fm_lds_budget(sizeof(T) == 4 ? 0 : 2), pol.gpaths,
                                a.npath_bucket, FM_WPE(T));
    if (g == -2) return hipErrorInvalidConfiguration;
    if (g < 0) return hipErrorInvalidValue;
    a.gp = 1 << g;
    a.bp = ed.bands[g];
    const size_t shm = a.path_bytes * a.gp;
    if (shm > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)k_matrices<T, SET>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)shm);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_matrices<T, SET>), dim3((unsigned)((a.npath_bucket + a.gp - 1) / a.gp)), dim3(FM_WAVE * 4), shm,
                       st, a);
    return hipGetLastError();
}

template <class T> hipError_t dispatch(KArgs &a, int set, const fm_launch &pol, hipStream_t st) {
    switch (set) {
        case 0: return launch_forward<T, 0>(a, pol, st);
        case 1: return launch_forward<T, 1>(a, pol, st);
        case FM_SET_SS: return launch_forward<T, FM_SET_SS>(a, pol, st);
        case FM_SET_SS + 1: return launch_forward<T, FM_SET_SS + 1>(a, pol, st);
        case FM_SET_SS + 2: return launch_forward<T, FM_SET_SS + 2>(a, pol, st);
    }
    return hipErrorInvalidValue;
}

// The policy of bucket b: the caller's, or the defaults (paths per workgroup by the LDS budget, one workgroup each).
fm_launch policy_of(const fm_launch *launch, int b) {
    fm_launch d;
    memset(&d, 0, sizeof d);
    return launch ? launch[b] : d;
}

const char *check_policy(const fm_launch &p) {
    if (p.gpaths != 0 && p.gpaths != 1 && p.gpaths != 2 && p.gpaths != 4 && p.gpaths != 8)
        return "launch policy: gpaths must be 0, 1, 2, 4 or 8";
    if (p.grid < -1) return "launch policy: grid must be -1, 0 or a number of workgroups";
    return nullptr;
}

int check_edge(const fm_edge *e) {
    const char *m = edge_problem(e);
    if (m) return set_err(FM_EINVAL, m);
    if (e->ilinit < 1 || e->ilinit > 3) return set_err(FM_EUNSUPPORTED, "edge: only K, L and M edges (ilinit 1..3)");
    return FM_OK;
}

}  // namespace

hipError_t fm::forward_matrices(int precision, const fm_edge &ed, const PathSrc &src, const int32_t *order, int first,
                                int npath, int nleg, void *keep, const fm_launch &pol, hipStream_t st) {
    KArgs a;
    memset(&a, 0, sizeof a);
    a.ed = ed;
    a.src = src;
    a.npath_bucket = npath;
    a.first = first;
    a.order = order;
    a.nleg = nleg;
    a.keep = keep;
    if (set_for(ed, nleg) == 0)
        return precision == 32 ? launch_matrices<float, 0>(a, pol, st) : launch_matrices<double, 0>(a, pol, st);
    return precision == 32 ? launch_matrices<float, 1>(a, pol, st) : launch_matrices<double, 1>(a, pol, st);
}

extern "C" {

const char *fm_last_error(void) { return g_err; }
const char *fm_version(void) { return "feffgpu_amd 0.1 (gfx950)"; }

size_t fm_keep_bytes(int32_t precision, const fm_edge *edge, int32_t nleg, int32_t npath) {
    if (!edge || nleg < 3 || nleg > 6 || npath <= 0 || (precision != 32 && precision != 64)) return 0;
    const int rows = edge->ilinit <= 1 ? keep_rows<0>(nleg) : keep_rows<1>(nleg);
    return (size_t)npath * (size_t)rows * (size_t)edge->E * 2 * (precision == 32 ? 4 : 8);
}

int32_t fm_set_lds_budget(int32_t kernel, int32_t kib) {
    if (kernel < 0 || kernel > 3 || kib < 16 || kib > 160) return -1;
    return (int32_t)(g_lds_budget[kernel].exchange((size_t)kib * 1024) / 1024);
}

int fm_cchi(const fm_edge *edge, int32_t precision, int32_t iorder, int32_t npath, int32_t nleg, const double *coords,
            const int64_t *ipots, void *cchi, double *reff, void *stream) {
    int rc = check_edge(edge);
    if (rc) return rc;
    if (iorder != 2) return set_err(FM_EUNSUPPORTED, "only iorder = 2 is implemented on the GPU");
    if (nleg < 2 || nleg > FM_MAX_LEGS) return set_err(FM_EINVAL, "nleg out of range 2..9");
    if (npath < 0) return set_err(FM_EINVAL, "npath < 0");
    if (npath == 0) return FM_OK;
    if (!coords || !ipots || !cchi) return set_err(FM_EINVAL, "NULL buffer");
    if (precision != 32 && precision != 64) return set_err(FM_EINVAL, "precision must be 32 or 64");
    const int set = set_for(*edge, nleg);
    KArgs a;
    memset(&a, 0, sizeof a);
    a.ed = *edge;
    a.src.mode = 0;
    a.npath_bucket = npath;
    a.first = 0;
    a.order = nullptr;
    a.src.nleg = nleg;
    a.src.coords = coords;
    a.src.ipots64 = ipots;
    a.src.nph1 = edge->nph1;
    a.cchi_out = cchi;
    a.reff_out = reff;
    a.edge_id = 0;
    a.nleg = nleg;
    hipStream_t st = (hipStream_t)stream;
    const fm_launch pol = policy_of(nullptr, 0);
    hipError_t e = precision == 32 ? dispatch<float>(a, set, pol, st) : dispatch<double>(a, set, pol, st);
    if (e == hipErrorInvalidValue) return set_err(FM_EINVAL, "fm_cchi: a path's tables do not fit one workgroup's LDS");
    return e == hipSuccess ? FM_OK : hip_err(e, "fm_cchi launch");
}

int fm_chi_fine(const fm_edge *edge, int32_t precision, int32_t npath, const void *cchi, const double *reff,
                const fm_grid *grid, void *chi, void *stream) {
    int rc = check_edge(edge);
    if (rc) return rc;
    if (npath < 0) return set_err(FM_EINVAL, "npath < 0");
    if (npath == 0) return FM_OK;
    if (!cchi || !reff || !grid || !chi || !grid->q || !grid->jq || !grid->fq) return set_err(FM_EINVAL, "NULL buffer");
    if (grid->S && grid->sstride < edge->E) return set_err(FM_EINVAL, "grid.sstride < E");
    if (precision != 32 && precision != 64) return set_err(FM_EINVAL, "precision must be 32 or 64");
    const size_t wb = align16((precision == 32 ? 4 : 8) * (size_t)edge->E) + align16(8 * (size_t)edge->E);
    const int wpb = WPB_MAX;
    const int blocks = (npath + wpb - 1) / wpb;
    hipStream_t st = (hipStream_t)stream;
    if (grid->S) {
        const dim3 g((unsigned)((npath + FM_WAVE - 1) / FM_WAVE), (unsigned)((grid->nk + DR * DW - 1) / (DR * DW)));
        if (grid->nk < 1) return FM_OK;
        if (precision == 32)
            hipLaunchKernelGGL(k_chi_dense<float>, g, dim3(FM_WAVE * DW), 0, st, *edge, npath, (const float *)cchi, reff,
                               *grid, (float *)chi);
        else
            hipLaunchKernelGGL(k_chi_dense<double>, g, dim3(FM_WAVE * DW), 0, st, *edge, npath, (const double *)cchi,
                               reff, *grid, (double *)chi);
    } else if (precision == 32)
        hipLaunchKernelGGL(k_chi_fine<float>, dim3(blocks), dim3(FM_WAVE * wpb), wb * wpb, st, *edge, npath,
                           (const float *)cchi, reff, *grid, (float *)chi, wb);
    else
        hipLaunchKernelGGL(k_chi_fine<double>, dim3(blocks), dim3(FM_WAVE * wpb), wb * wpb, st, *edge, npath,
                           (const double *)cchi, reff, *grid, (double *)chi, wb);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FM_OK : hip_err(e, "fm_chi_fine launch");
}

int fm_chi_paths(const fm_edge *edges, int32_t nedge, const fm_paths *paths, const fm_grid *grid, int32_t precision,
                 int32_t iorder, const int32_t *order, int32_t nbucket, const int32_t *bucket_offset,
                 const int32_t *bucket_kind, const int32_t *bucket_edge, const int32_t *bucket_nleg, int32_t nseg,
                 const int32_t *seg_ptr, const int32_t *seg_paths, double *chi_seg, void *chi_path, double *reff,
                 const fm_launch *launch, void *stream) {
    return fm_chi_paths_overlap(edges, nedge, paths, grid, precision, iorder, order, nbucket, bucket_offset, bucket_kind,
                                bucket_edge, bucket_nleg, nseg, seg_ptr, seg_paths, chi_seg, chi_path, reff, launch,
                                nullptr, stream);
}

int fm_chi_paths_overlap(const fm_edge *edges, int32_t nedge, const fm_paths *paths, const fm_grid *grid,
                         int32_t precision, int32_t iorder, const int32_t *order, int32_t nbucket,
                         const int32_t *bucket_offset, const int32_t *bucket_set, const int32_t *bucket_edge,
                         const int32_t *bucket_nleg, int32_t nseg, const int32_t *seg_ptr, const int32_t *seg_paths,
                         double *chi_seg, void *chi_path, double *reff, const fm_launch *launch, fm_overlap *overlap,
                         void *stream) try {
    if (nedge < 1 || nedge > FM_MAX_EDGE) return set_err(FM_EINVAL, "nedge out of range 1..4");
    for (int i = 0; i < nedge; ++i) {
        int rc = check_edge(&edges[i]);
        if (rc) return rc;
    }
    if (iorder != 2) return set_err(FM_EUNSUPPORTED, "only iorder = 2 is implemented on the GPU");
    if (!paths || !grid || !chi_path) return set_err(FM_EINVAL, "NULL paths, grid or chi_path");
    if (precision != 32 && precision != 64) return set_err(FM_EINVAL, "precision must be 32 or 64");
    if (paths->nmax < 2 || paths->nmax > FM_MAX_LEGS) return set_err(FM_EINVAL, "nmax out of range 2..9");
    if (grid->nk < 1) return set_err(FM_EINVAL, "empty grid");
    for (int i = 0; i < nedge; ++i)
        if (grid->S && grid->sstride < edges[i].E) return set_err(FM_EINVAL, "grid.sstride < E");
    if (nbucket > 0 && (!bucket_offset || !bucket_set || !bucket_nleg)) return set_err(FM_EINVAL, "NULL bucket arrays");
    hipStream_t st = (hipStream_t)stream;
    Lanes lanes(overlap, st, nbucket);
    const std::vector<int> lane = lanes_of(nbucket, bucket_offset, bucket_nleg, lanes.n);
    for (int b = 0; b < nbucket; ++b) {
        const int cnt = bucket_offset[b + 1] - bucket_offset[b];
        if (cnt <= 0) continue;
        const int kind = bucket_set[b];
        if (kind < 0 || kind > 2) return set_err(FM_EINVAL, "bucket kind out of range 0..2");
        KArgs a;
        memset(&a, 0, sizeof a);
        a.src.mode = 1;
        a.npath_bucket = cnt;
        a.first = bucket_offset[b];
        a.order = order;
        a.src.P = *paths;
        a.G = *grid;
        a.chi_path = chi_path;
        a.reff_out = reff;
        a.edge_id = bucket_edge ? bucket_edge[b] : 0;
        if (a.edge_id < 0 || a.edge_id >= nedge) return set_err(FM_EINVAL, "bucket edge out of range");
        a.ed = edges[a.edge_id];
        a.nleg = bucket_nleg[b];
        if (a.nleg < 2 || a.nleg > paths->nmax) return set_err(FM_EINVAL, "bucket nleg out of range 2..nmax");
        if ((kind == FM_BUCKET_SS) != (a.nleg == 2)) return set_err(FM_EINVAL, "bucket kind does not match its nleg");
        if ((kind == FM_BUCKET_K_MS) != (a.ed.ilinit <= 1) && kind != FM_BUCKET_SS)
            return set_err(FM_EINVAL, "bucket kind does not match its edge");
        const int set = set_for(a.ed, a.nleg);
        const fm_launch pol = policy_of(launch, b);
        if (const char *m = check_policy(pol)) return set_err(FM_EINVAL, m);
        if (pol.keep && kind != FM_BUCKET_SS && a.nleg >= 3 && a.nleg <= 6) {
            if (pol.keep_bytes < fm_keep_bytes(precision, &a.ed, a.nleg, cnt))
                return set_err(FM_EINVAL, "fm_chi_paths: keep_bytes smaller than fm_keep_bytes for the bucket");
            a.keep = pol.keep;
        }
        hipError_t e = precision == 32 ? dispatch<float>(a, set, pol, lanes.at(lane[b]))
                                        : dispatch<double>(a, set, pol, lanes.at(lane[b]));
        if (e == hipErrorInvalidValue) return set_err(FM_EINVAL, "fm_chi_paths: the bucket's paths do not fit one workgroup's LDS");
        if (e == hipErrorInvalidConfiguration)
            return set_err(FM_EINVAL, "fm_chi_paths: the launch policy's gpaths has no band plan or does not fit one CU's LDS");
        if (e != hipSuccess) return hip_err(e, "fm_chi_paths launch");
    }
    if (hipError_t e = lanes.join()) return hip_err(e, "fm_chi_paths side streams");
    if (chi_seg && nseg > 0) {
        if (!seg_ptr || !seg_paths) return set_err(FM_EINVAL, "NULL segment lists");
        if (precision == 32)
            launch_segment_sum(nseg, grid->nk, seg_ptr, seg_paths, paths->deg, (const float *)chi_path, chi_seg, st);
        else
            launch_segment_sum(nseg, grid->nk, seg_ptr, seg_paths, paths->deg, (const double *)chi_path, chi_seg, st);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return hip_err(e, "segment sum launch");
    }
    return FM_OK;
} catch (const std::exception &) {
    return set_err(FM_EINVAL, "fm_chi_paths: out of host memory");
}

}  // extern "C"
