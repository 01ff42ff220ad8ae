// The adjoint of multiple-scattering paths of 3-6 legs: d loss / d coordinates (GPUPathStage.cchi) or d loss /
// d positions of a path list, the gradient that feffgpu obtains by autograd through src/feffgpu/stage.py:147-388 and
// the gather of src/feffgpu/exafs/forward.py:153-163.
//
// It starts from the scattering matrices F_s (their independent entries, per energy) that the forward call kept, or
// that k_matrices (fm_forward.hip) rebuilds in the workspace. ptrac = tr(T F_{n-1} ... F_1) is a polynomial in the
// entries, so for every real parameter theta of the geometry (leg lengths, angles, eta) the derivative
// D_theta = d ptrac / d theta is formed without the upstream gradient, and the loss gradient is Re(pbc D_theta) with
// pbc = conj(dL/dptrac), summed over the energies. Five kernels:
//   k_setup     the leg geometry (FP64) and the termination's rotation rows, into a record per path.
//   k_chain     one wavefront per (path, 64 energies): the chain both ways, cchi, D of the termination and of every
//               eta, and per scatterer K_s = Pre_s U_s folded onto the independent entries (Pre_s = F_{s-1} ... F_1,
//               U_s = T F_{n-1} ... F_{s+1}). No partial-wave loop: every lane does the same work, and what belongs
//               to the path is wave-uniform.
//   k_pbc       one wavefront per path: the fine grid's adjoint (or the given dL/dcchi), pbc, and the sums over the
//               energies of k_chain's derivatives and the cfac terms.
//   k_stream    (path, scatterer) units: the rotation tables of the unit's leg, then per energy the stream over the
//               partial waves that contracts K_s with the derivatives of F_s in its two leg lengths and its angle,
//               times pbc, summed over the energies.
//   k_geometry  the per-leg gradients through the FP64 leg geometry (dual numbers), to the path's coordinates.
// The stream is most of the arithmetic. Alone it holds K and the two recursions (about 180 registers; 365 with the
// chain's matrices, one wavefront per SIMD), so two wavefronts share a SIMD; its units are many and small, which
// balances the very uneven numbers of partial waves per energy (5 to 29 on a K edge); and its sums need no per-energy
// slots in memory. K costs one write and one read of as many bytes as the kept matrices. Against the one-kernel sweep
// that this replaces (MI355X, FP32, us): 94 304 K-edge paths of 3 legs, 3570 -> 2470 (chain 750 at 3.9 TB/s, stream 1046
// with the vector pipes 88 % busy, pbc 537, setup 71, geometry 66); a NiO box of 2-4 legs, whole step, 21.6 -> 17.0 ms;
// the same in FP64 on a smaller box 2.30 -> 1.63 ms.
//
// The single-precision sums of this file keep their roundings to the last bit from one layout of the work to the next:
// where the compiler's choice of the product that a fused multiply-add takes depends on what it shares with its
// neighbours (SeedX, chain_step's S == 2), the multiply-adds are written out.
#include <hip/hip_runtime.h>
#include <string.h>

#include <type_traits>

#include "fm_device.h"
#include "fm_grad.h"
#include "fm_internal.h"
#include "fm_path.h"

using namespace fm;

size_t fm_lds_budget(int kernel);

namespace {

// ------------------------------------------------------------------------------------------------ the workspace
// Per path a record of doubles: cos/sin of beta and beta/2 of every leg, the leg lengths (bohr), the potential of
// every atom, the path length and the product of the leg lengths; the sums over the energies of k_chain's derivatives
// (eta_1..eta_n, the termination's three), of the cfac terms (a1, a2) and dL/dreff; k_stream's three sums per
// scatterer.
__host__ __device__ constexpr int rec_trig(int) { return 0; }
__host__ __device__ constexpr int rec_r(int n) { return 4 * n; }
__host__ __device__ constexpr int rec_pot(int n) { return 5 * n; }
__host__ __device__ constexpr int rec_len_r(int n) { return 6 * n; }        // R, prod r
__host__ __device__ constexpr int rec_sum(int n) { return 6 * n + 2; }
__host__ __device__ constexpr int rec_stream(int n) { return 7 * n + 8; }
__host__ __device__ constexpr int rec_len(int n) { return 10 * n + 5; }
// and one of T: cos/sin of eta and 2 eta per leg, the termination's rotation rows 1..4 and their beta derivatives.
__host__ __device__ constexpr int rt_w(int n) { return 4 * n; }
__host__ __device__ constexpr int rt_len(int n) { return 4 * n + 8 * FM_NREP; }
// and per energy cchi (pbc after k_pbc) and k_chain's n + 3 complex derivatives, [row][energy].
__host__ __device__ constexpr int slot_rows(int n) { return n + 4; }

// K: [group of 16 paths][scatterer][band of 4 energies][entry][16 paths x 4 energies] complex T, so that a wavefront
// of k_stream (16 paths, 4 energies) reads whole lines, and the four paths of k_chain's workgroup write them. The
// bands count down from the last energy, as k_stream takes them.
constexpr int KG = 16, KB = 4;
__host__ __device__ inline size_t k_group(int rows, int E) { return (size_t)rows * ((E + KB - 1) / KB) * (KG * KB); }
__device__ __forceinline__ int k_band(int e, int E) { return (E - 1 - e) / KB; }
__device__ __forceinline__ int k_slot(int e, int E) { return KB - 1 - (E - 1 - e) % KB; }

template <class T> struct MArgs {
    fm_edge ed;
    int npath, first, edge_id;
    const int32_t *order;
    PathSrc src;
    const T *gcchi;
    const double *greff;
    fm_grid G;
    const int32_t *segment;
    const double *gseg;
    const T *gpath;
    double *gcoord;
    int nslot, nk, nleg;
    const T *F;               // the launch's kept matrices, its first path first
    T *K;
    double *rec;
    T *rt;
    T *slot;
    int once;                 // 1: the trip count of a loop that keeps chain_step's stores in a block of their own
    int units;                // k_stream: (path, scatterer) units per workgroup
    size_t wave_bytes, off_amp, off_ang, off_cb, off_qs;   // k_pbc: LDS of one wavefront
    size_t unit_bytes;        // k_stream: LDS of one unit's tables
};

// ------------------------------------------------------------------------------------------------ the setup
// Sixteen paths per workgroup, a group of 16 lanes each; then the termination's rotation rows il = 1..4 of leg n, one
// (path, representative) per thread.
template <class T, int SET>
__global__ __launch_bounds__(256) void k_setup(MArgs<T> a) {
    __shared__ PathLDS gs[16];
    const int t = threadIdx.x, n = a.nleg;
    const fm_edge &ed = a.ed;
    {
        const int q = blockIdx.x * 16 + t / 16, lane = t & 15;
        const int s0 = q < a.npath ? q : blockIdx.x * 16;
        const int p = a.order ? a.order[a.first + s0] : a.first + s0;
        PathLDS &g = gs[t / 16];
        int ei;
        load_path_group(a.src, p, g, ei, n, lane, true);
        if (q < a.npath) {
            double *rec = a.rec + (size_t)q * rec_len(n);
            T *rt = a.rt + (size_t)q * rt_len(n);
            if (lane < n) {
                const int j = lane + 1;
                rec[rec_trig(n) + 4 * lane] = g.cb[j];
                rec[rec_trig(n) + 4 * lane + 1] = g.sb[j];
                rec[rec_trig(n) + 4 * lane + 2] = g.ch[j];
                rec[rec_trig(n) + 4 * lane + 3] = g.sh[j];
                rec[rec_r(n) + lane] = g.r[j];
                rec[rec_pot(n) + lane] = (double)g.ipot[lane];
                rt[4 * lane] = (T)g.c1[j];
                rt[4 * lane + 1] = (T)g.s1[j];
                rt[4 * lane + 2] = (T)g.c2[j];
                rt[4 * lane + 3] = (T)g.s2[j];
            }
            if (lane == 0) {
                rec[rec_len_r(n)] = g.R;
                rec[rec_len_r(n) + 1] = g.prod_r;
            }
        }
    }
    __syncthreads();
    for (int x = t; x < 16 * FM_NREP; x += 256) {
        constexpr PairDef PD = pairdef(SET);
        const int u = x / FM_NREP, k = x - u * FM_NREP, q = blockIdx.x * 16 + u;
        if (q >= a.npath) continue;
        int m1 = 0, m2 = 0;
#pragma unroll
        for (int r = 0; r < FM_NREP; ++r)
            if (r == k) { m1 = PD.m1[r]; m2 = PD.m2[r]; }
        const int am1 = m1 < 0 ? -m1 : m1, am2 = m2 < 0 ? -m2 : m2;
        RotCoef<4> rc;
        rc.fetch(ed, 1, ed.L1 < 4 ? ed.L1 : 4, (m1 + 3) * 7 + (m2 + 3), am1 * 4 + am2);
        const PathLDS &g = gs[u];
        const double c = g.cb[n], sn = g.sb[n], c2 = g.ch[n], s2 = g.sh[n];
        double d1 = 0.0, d0 = 0.0, t1 = 0.0, t0 = 0.0;
        T *const w = a.rt + (size_t)q * rt_len(n) + rt_w(n) + k;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double d, td;
            if (v <= 2) {
                d = dseed(v, m1, m2, c, sn, c2, s2);
                td = dseed_db(v, m1, m2, c, sn, c2, s2);
            } else {
                const double a1 = rc.c0[v] * c - rc.c1[v];
                d = a1 * d1 - rc.c2[v] * d0;
                td = a1 * t1 - rc.c0[v] * sn * d1 - rc.c2[v] * t0;
            }
            d0 = d1; d1 = d;
            t0 = t1; t1 = td;
            w[v * FM_NREP] = (T)(d * rc.nr[v]);
            w[(4 + v) * FM_NREP] = (T)(td * rc.nr[v]);
        }
    }
}

// ------------------------------------------------------------------------------------------------ one row
// Bit 2 aa + bb set: some representative of an NR x NC block has Hankel columns (aa + 1, bb + 1).
template <int SET, int NR, int NC>
__host__ __device__ constexpr unsigned group_mask() {
    constexpr PairDef PD = pairdef(SET);
    unsigned m = 0;
    for (int k = 0; k < FM_NREP; ++k)
        if (PD.ri[k] < NR && PD.rj[k] < NC) m |= 1u << (2 * (PD.a[k] - 1) + PD.b[k] - 1);
    return m;
}

// One partial-wave row of a block's tangents contracted with K, accumulated as complex derivatives. y, yd: the
// gamtl leg's factors and their tangents without the row's t-matrix factor t, which scales the row's three sums once.
template <class T, int SET, int NR, int NC, class WRow>
__device__ __forceinline__ void bwd_row_c(const cx<T> (&K)[FM_NREP], const cx<T> (&xa)[3], const cx<T> (&xd)[3],
                                          const cx<T> (&y)[2], const cx<T> (&yd)[2], cx<T> t, const WRow &w,
                                          const WRow &wd, cx<T> &dX, cx<T> &dY, cx<T> &dB) {
    constexpr PairDef PD = pairdef(SET);
    constexpr unsigned used = group_mask<SET, NR, NC>();
    const cx<T> zero = mk<T>(T(0), T(0));
    cx<T> Q[3][2], Qd[3][2];
#pragma unroll
    for (int aa = 0; aa < 3; ++aa) Q[aa][0] = Q[aa][1] = Qd[aa][0] = Qd[aa][1] = zero;
#pragma unroll
    for (int k = 0; k < FM_NREP; ++k)
        if (PD.ri[k] < NR && PD.rj[k] < NC) {
            const int aa = PD.a[k] - 1, bb = PD.b[k] - 1;
            rfma(Q[aa][bb], K[k], w[k]);
            rfma(Qd[aa][bb], K[k], wd[k]);
        }
    // dB: sum Qd[aa][bb] xa[aa] y[bb]; dY: sum Q[aa][bb] xa[aa] yd[bb]; dX: sum Q[aa][bb] xd[aa] y[bb]
    cx<T> sB = zero, sY = zero, sX = zero;
#pragma unroll
    for (int bb = 0; bb < 2; ++bb) {
        if (!((used >> bb) & 0x15u)) continue;
        cx<T> rd = zero, r = zero, v = zero;
#pragma unroll
        for (int aa = 0; aa < 3; ++aa)
            if ((used >> (2 * aa + bb)) & 1u) {
                cfma4(rd, Qd[aa][bb], xa[aa]);
                cfma4(r, Q[aa][bb], xa[aa]);
                cfma4(v, Q[aa][bb], xd[aa]);
            }
        cfma4(sB, y[bb], rd);
        cfma4(sY, yd[bb], r);
        cfma4(sX, y[bb], v);
    }
    cfma4(dB, t, sB);
    cfma4(dY, t, sY);
    cfma4(dX, t, sX);
}

// ------------------------------------------------------------------------------------------------ the chain
// A lane's outputs, buffer stores that drop the lanes past the last energy (their offset is past the end): the
// derivative slots eta_1..eta_n (0..n-1) and the termination's three (n..n+2) of the lane's energy, and entry q of
// scatterer S's K.
template <class T> struct Slots {
    __amdgpu_buffer_rsrc_t rs, ks;
    uint32_t lo, klo;     // the lane's energy in slot row 1; its (path, energy) slot in the group's K
    int sbytes, band, nb, once;
    __device__ __forceinline__ void put(int k, cx<T> x) const { buf_st(rs, lo, k * sbytes, x); }
};

// F(i, j) of a block from its representatives, with the row phase: ph[i] sg Ft[idx[i][j]]
template <class T, int SET>
__device__ __forceinline__ cx<T> fent(const cx<T> (&Ft)[FM_NREP], const cx<T> (&ph)[6], int i, int j) {
    constexpr PairDef PD = pairdef(SET);
    return ph[i] * Ft[PD.idx[i][j]] * T(PD.sg[i][j]);
}

// fent with its multiply-adds written out
template <class T, int SET>
__device__ __forceinline__ cx<T> fent_fma(const cx<T> (&Ft)[FM_NREP], const cx<T> (&ph)[6], int i, int j) {
    constexpr PairDef PD = pairdef(SET);
    const cx<T> f = Ft[PD.idx[i][j]];
    if (lamdef(SET).M[i] == 0) return f * T(PD.sg[i][j]);
    return mk<T>(fma(f.r, ph[i].r, -(f.i * ph[i].i)), fma(f.i, ph[i].r, f.r * ph[i].i)) * T(PD.sg[i][j]);
}

// Pre_S = F_{S-1} ... F_1 (L x L0, with the row phases) from the kept representatives; S >= 2.
template <class T, int SET, int NL, int S, bool FMA = false>
__device__ __forceinline__ void prefix(const PathLDS &g, const cx<T> (&F)[NL - 1][FM_NREP],
                                       cx<T> (&P)[lamdef(SET).L][lamdef(SET).L0]) {
    constexpr int L = lamdef(SET).L, L0 = lamdef(SET).L0;
    cx<T> ph[6];
    row_phases<T, SET>(ph, g, 2);
#pragma unroll
    for (int i = 0; i < L; ++i)
#pragma unroll
        for (int b = 0; b < L0; ++b) P[i][b] = FMA ? fent_fma<T, SET>(F[0], ph, i, b) : fent<T, SET>(F[0], ph, i, b);
#pragma unroll
    for (int t = 2; t < S; ++t) {   // Pre_{t+1} = F_t Pre_t
        row_phases<T, SET>(ph, g, t + 1);
#pragma unroll
        for (int b = 0; b < L0; ++b) {
            cx<T> col[L];
#pragma unroll
            for (int j = 0; j < L; ++j) col[j] = P[j][b];
#pragma unroll
            for (int i = 0; i < L; ++i) {
                cx<T> acc = mk<T>(T(0), T(0));
#pragma unroll
                for (int j = 0; j < L; ++j) cfma4(acc, fent<T, SET>(F[t - 1], ph, i, j), col[j]);
                P[i][b] = acc;
            }
        }
    }
}

// One chain step (scatterer S; NR x NC block): K and the eta derivative from Pre_S and U, then U <- U F_S (unless
// S = 1).
template <class T, int SET, int NL, int S>
__device__ __forceinline__ void chain_step(const PathLDS &g, const cx<T> (&F)[NL - 1][FM_NREP],
                                           cx<T> (&U)[lamdef(SET).L0][lamdef(SET).L], Slots<T> ds) {
    constexpr LamDef D = lamdef(SET);
    constexpr PairDef PD = pairdef(SET);
    constexpr int L = D.L, L0 = D.L0;
    constexpr int NR = S == NL - 1 ? L0 : L, NC = S == 1 ? L0 : L;
    cx<T> ph[6];
    row_phases<T, SET>(ph, g, S + 1);
    cx<T> K[FM_NREP];
    {
        cx<T> P[L][L0];
        if constexpr (S >= 2) prefix<T, SET, NL, S, (S == 2 && NL >= 4)>(g, F, P);
#pragma unroll
        for (int k = 0; k < FM_NREP; ++k) K[k] = mk<T>(T(0), T(0));
        // K from Pre_S and U; the eta_{S+1} derivative -i sum_{l1,l2} M[l1] h(l1, l2) F_S(l1, l2) on the way
        cx<T> de = mk<T>(T(0), T(0));
#pragma unroll
        for (int l2 = 0; l2 < NC; ++l2) {
#pragma unroll
            for (int l1 = 0; l1 < NR; ++l1) {
                cx<T> m = mk<T>(T(0), T(0));
                if constexpr (S >= 2) {
#pragma unroll
                    for (int a = 0; a < L0; ++a) cfma4(m, P[l2][a], U[a][l1]);
                } else {
                    m = U[l2][l1];
                }
                cx<T> h = m * ph[l1];
                if (S == 2 && NL >= 4 && D.M[l1] != 0) {
                    h.r = fma(m.r, ph[l1].r, -(m.i * ph[l1].i));
                    h.i = D.M[l1] < 0 && D.M[l2] != 0 ? fma(m.r, ph[l1].i, m.i * ph[l1].r) : fma(m.i, ph[l1].r, m.r * ph[l1].i);
                }
                if (PD.sg[l1][l2] > 0) K[PD.idx[l1][l2]] = K[PD.idx[l1][l2]] + h;
                else K[PD.idx[l1][l2]] = K[PD.idx[l1][l2]] - h;
                if (D.M[l1] != 0) cfma4(de, h * T(PD.sg[l1][l2] * D.M[l1]), F[S - 1][PD.idx[l1][l2]]);
            }
        }
        ds.put(S, mk<T>(de.i, -de.r));
        if constexpr (S > 1) {
#pragma unroll
            for (int a = 0; a < L0; ++a) {
                cx<T> row[6];
#pragma unroll
                for (int i = 0; i < 6; ++i) row[i] = (i < NR) ? U[a][i] * ph[i] : mk<T>(T(0), T(0));
#pragma unroll
                for (int j = 0; j < L; ++j) {
                    cx<T> v = mk<T>(T(0), T(0));
                    if (j < NC) {
#pragma unroll
                        for (int i = 0; i < NR; ++i) {
                            const cx<T> f = F[S - 1][PD.idx[i][j]];
                            if (PD.sg[i][j] > 0) cfma4(v, row[i], f); else cfma4(v, row[i], mk<T>(-f.r, -f.i));
                        }
                    }
                    U[a][j] = v;
                }
            }
        }
    }
    constexpr KeepList KL = keep_list(SET, NR, NC);
    const uint32_t ko = ds.klo + (uint32_t)((ds.nb * keep_off<SET>(NL, S) + ds.band * KL.n) * (KG * KB) * (int)sizeof(cx<T>));
#pragma unroll 1
    for (int it = 0; it < ds.once; ++it) {
#pragma unroll
        for (int q = 0; q < KL.n; ++q) buf_st(ds.ks, ko, q * (KG * KB) * (int)sizeof(cx<T>), K[KL.k[q]]);
    }
}

template <class T, int SET, int NL, int S>
__device__ __forceinline__ void chain_steps(const PathLDS *gs, int wid, const cx<T> (&F)[NL - 1][FM_NREP],
                                            cx<T> (&U)[lamdef(SET).L0][lamdef(SET).L], Slots<T> ds) {
    chain_step<T, SET, NL, S>(gs[wid], F, U, ds);
    // the phases are read again at every step instead of held (an index the compiler cannot see through)
    asm volatile("" : "+s"(wid));
    if constexpr (S > 1) chain_steps<T, SET, NL, S - 1>(gs, wid, F, U, ds);
}

// The kept matrices of scatterers S..NL-1 from the lane's rows (the first scatterer's block is L x L0, the last's
// L0 x L, the others L x L).
template <class T, int SET, int NL, int S>
__device__ __forceinline__ void keep_loads(const T *kp, int E, cx<T> (&F)[NL - 1][FM_NREP]) {
    constexpr int L = lamdef(SET).L, L0 = lamdef(SET).L0;
    const T *b = kp + (size_t)2 * E * keep_off<SET>(NL, S);
    if constexpr (S == 1) keep_load<T, SET, L, L0>(b, E, F[S - 1]);
    else if constexpr (S == NL - 1) keep_load<T, SET, L0, L>(b, E, F[S - 1]);
    else keep_load<T, SET, L, L>(b, E, F[S - 1]);
    if constexpr (S < NL - 1) keep_loads<T, SET, NL, S + 1>(kp, E, F);
}

// The chain at energy ee from the scattering matrices F of every scatterer: returns cchi and stores the complex
// derivatives of ptrac and K in ds.
template <class T, int SET, int NL>
__device__ __forceinline__ cx<T> chain_energy(const fm_edge &ed, const PathLDS *gs, int wid, const T *Wn, const T *Wdn, int ee,
                                              Slots<T> ds, const cx<T> (&F)[NL - 1][FM_NREP]) {
    const PathLDS &g = gs[wid];
    constexpr LamDef D = lamdef(SET);
    constexpr PairDef PD = pairdef(SET);
    constexpr int L = D.L, L0 = D.L0;
    const int E = ed.E;
    // read ahead of Pre_n, whose work hides their latency: the termination's channel weights of rows 1..4 (a row
    // without a channel reads channel 0's and does not use it) and ck
    const cx<T> ck = mk<T>((T)ed.ck[2 * ee], (T)ed.ck[2 * ee + 1]);
    const T *chw = TL<T>::chw(ed);
    int chan[4];
    cx<T> wraw[4];
#pragma unroll
    for (int r = 1; r <= 4; ++r) {
        int c = -1;
        for (int q = 0; q < ed.nchan; ++q)
            if (ed.chan_il[q] == r) c = q;
        chan[r - 1] = c;
        const size_t o = ((size_t)(c >= 0 ? c : 0) * E + ee) * 2;
        wraw[r - 1] = mk<T>(chw[o], chw[o + 1]);
    }
    // Pre_n (L0 x L0)
    cx<T> Pn[L0][L0];
    {
        cx<T> P[L][L0];
        prefix<T, SET, NL, NL - 1>(g, F, P);
        cx<T> ph[6];
        row_phases<T, SET>(ph, g, NL);
#pragma unroll
        for (int i = 0; i < L0; ++i)
#pragma unroll
            for (int b = 0; b < L0; ++b) {
                cx<T> acc = mk<T>(T(0), T(0));
#pragma unroll
                for (int j = 0; j < L; ++j) cfma4(acc, fent<T, SET>(F[NL - 2], ph, i, j), P[j][b]);
                Pn[i][b] = acc;
            }
    }
    // termination: T with its tangents against K_T[a][b] = Pn[b][a] ph1[a]
    cx<T> U[L0][L];
    cx<T> ptrac = mk<T>(T(0), T(0));
    {
        cx<T> ph[6];
        row_phases<T, SET>(ph, g, 1);
        cx<T> K[FM_NREP];
#pragma unroll
        for (int k = 0; k < FM_NREP; ++k) K[k] = mk<T>(T(0), T(0));
#pragma unroll
        for (int a = 0; a < L0; ++a)
#pragma unroll
            for (int b = 0; b < L0; ++b) {
                const cx<T> h = Pn[b][a] * ph[a];
                if (PD.sg[a][b] > 0) K[PD.idx[a][b]] = K[PD.idx[a][b]] + h;
                else K[PD.idx[a][b]] = K[PD.idx[a][b]] - h;
            }
        const int *lm = ed.lmax + ee;
        const int lx1 = max(lm[(size_t)g.ipot[0] * E], lm[(size_t)g.ipot[1] * E]) + 1;
        const int lxn = max(lm[(size_t)g.ipot[NL - 1] * E], lm[(size_t)g.ipot[NL] * E]) + 1;
        Hank3T<T> X;
        Hank2T<T> Y;
        X.init(minus_i_over(ck * (T)g.r[1]), (T)g.r[1]);
        Y.init(minus_i_over(ck * (T)g.r[NL]), (T)g.r[NL]);
        cx<T> Tt[FM_NREP];
#pragma unroll
        for (int k = 0; k < FM_NREP; ++k) Tt[k] = mk<T>(T(0), T(0));
        cx<T> dX = mk<T>(T(0), T(0)), dY = dX, dB = dX;
        cx<T> xa[3], xd[3], ya[2], yd[2];
#pragma unroll
        for (int r = 1; r <= 4; ++r) {
            X.seed_row(r, xa, xd, r <= lx1);
            if (r < 4) Y.seed_row(r, ya, yd, r <= lxn); else Y.step(r, ya, yd, r <= lxn);
            if (chan[r - 1] >= 0) {
                const cx<T> w = wraw[r - 1] * T(2 * r - 1);
                accum_row<T, SET, L0, L0>(Tt, xa, ya[0] * w, ya[1] * w, Wn + (size_t)r * FM_NREP);
                bwd_row_c<T, SET, L0, L0>(K, xa, xd, ya, yd, w, Wn + (size_t)r * FM_NREP, Wdn + (size_t)r * FM_NREP,
                                          dX, dY, dB);
            }
        }
        ds.put(NL, dX);
        ds.put(NL + 1, dY);
        ds.put(NL + 2, dB);
        cx<T> de = mk<T>(T(0), T(0));
#pragma unroll
        for (int a = 0; a < L0; ++a)
#pragma unroll
            for (int b = 0; b < L; ++b) {
                const cx<T> t = (b < L0) ? ph[a] * Tt[PD.idx[a][b]] * T(PD.sg[a][b]) : mk<T>(T(0), T(0));
                U[a][b] = t;
                if (b < L0) {
                    const cx<T> tp = t * Pn[b][a];
                    ptrac = ptrac + tp;
                    if (D.M[a] != 0) rfma(de, tp, T(D.M[a]));
                }
            }
        ds.put(0, mk<T>(de.i, -de.r));
    }
    chain_steps<T, SET, NL, NL - 1>(gs, wid, F, U, ds);
    return ptrac * cfac_at<T>(ed, g, ee, NL);
}

// One wavefront per (path, 64 energies), four per workgroup, no workgroup barrier.
template <class T, int SET, int NL, int WPE>
__global__ __launch_bounds__(FM_WAVE * 4) __attribute__((amdgpu_waves_per_eu(WPE))) void k_chain(MArgs<T> a) {
    __shared__ PathLDS gs[4];
    __shared__ T ws[4][10 * FM_NREP];
    constexpr int n = NL;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FM_WAVE), lane = lane_id();
    const fm_edge &ed = a.ed;
    const int E = ed.E, nchunk = (E + FM_WAVE - 1) / FM_WAVE;
    const int w = blockIdx.x * 4 + wid, s0 = w / nchunk;
    if (s0 >= a.npath) return;
    PathLDS &g = gs[wid];
    {
        const double *rec = a.rec + (size_t)s0 * rec_len(n);
        const T *rt = a.rt + (size_t)s0 * rt_len(n);
        for (int x = lane; x < 4 * FM_NREP; x += FM_WAVE) {
            ws[wid][FM_NREP + x] = rt[rt_w(n) + x];
            ws[wid][6 * FM_NREP + x] = rt[rt_w(n) + 4 * FM_NREP + x];
        }
        if (lane < n) {
            g.c1[lane + 1] = rt[4 * lane];
            g.s1[lane + 1] = rt[4 * lane + 1];
            g.c2[lane + 1] = rt[4 * lane + 2];
            g.s2[lane + 1] = rt[4 * lane + 3];
            g.r[lane + 1] = rec[rec_r(n) + lane];
            g.ipot[lane] = (int)rec[rec_pot(n) + lane];
        }
        if (lane == 0) {
            g.ipot[n] = (int)rec[rec_pot(n)];
            g.R = rec[rec_len_r(n)];
            g.prod_r = rec[rec_len_r(n) + 1];
        }
        wave_sync();
    }
    const int e0 = (w - s0 * nchunk) * FM_WAVE;
    const bool on = e0 + lane < E;
    const int ee = on ? e0 + lane : E - 1;
    constexpr int rows = keep_rows<SET>(NL);
    cx<T> *const slot = reinterpret_cast<cx<T> *>(a.slot) + (size_t)s0 * slot_rows(n) * E;
    const size_t kg = k_group(rows, E);
    const Slots<T> ds{slice_rsrc(reinterpret_cast<unsigned char *>(slot), (size_t)slot_rows(n) * E * sizeof(cx<T>)),
                      slice_rsrc(reinterpret_cast<unsigned char *>(a.K + (size_t)(s0 / KG) * kg * 2), kg * sizeof(cx<T>)),
                      on ? (uint32_t)((E + ee) * sizeof(cx<T>)) : 0x40000000u,
                      on ? (uint32_t)(((s0 % KG) * KB + k_slot(ee, E)) * sizeof(cx<T>)) : 0x40000000u,
                      E * (int)sizeof(cx<T>), k_band(ee, E), (E + KB - 1) / KB, a.once};
    cx<T> F[NL - 1][FM_NREP];
    if (a.F) {     // never NULL: the branch keeps the loads in a block of their own, before everything that uses them
        keep_loads<T, SET, NL, 1>(a.F + ((size_t)s0 * rows * E + ee) * 2, E, F);
    } else {
#pragma unroll
        for (int s = 0; s < NL - 1; ++s)
#pragma unroll
            for (int k = 0; k < FM_NREP; ++k) F[s][k] = mk<T>(T(0), T(0));
    }
    const cx<T> c = chain_energy<T, SET, NL>(ed, gs, wid, ws[wid], ws[wid] + 5 * FM_NREP, ee, ds, F);
    if (on) slot[ee] = c;
}

// ------------------------------------------------------------------------------------------------ pbc
// Sums of up to 16 values per lane over the wavefront: each step folds half of the values onto the other half of the
// lanes, so 17 exchanges give all 16 sums (lane l holds sum (l >> 2) in every fourth lane), in a fixed order.
__device__ __forceinline__ double wave_sum16(double (&v)[16]) {
    const int lane = lane_id();
#pragma unroll
    for (int h = 8, off = 32; h >= 1; h >>= 1, off >>= 1) {
        const bool up = lane & off;
#pragma unroll
        for (int k = 0; k < h; ++k) {
            const double mine = up ? v[k + h] : v[k], theirs = up ? v[k] : v[k + h];
            v[k] = mine + __shfl_xor(theirs, off, FM_WAVE);
        }
    }
    double s = v[0];
    s += __shfl_xor(s, 2, FM_WAVE);
    s += __shfl_xor(s, 1, FM_WAVE);
    return s;
}

// One wavefront per path, four per workgroup, no workgroup barrier (a wavefront without a path returns): few registers
// and a few KB of LDS, so that several wavefronts share a SIMD and hide the latencies this work consists of.
template <class T, int NL>
__global__ __launch_bounds__(FM_WAVE * 4) void k_pbc(MArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wid = threadIdx.x / FM_WAVE, lane = lane_id();
    const int s0 = blockIdx.x * 4 + wid;
    if (s0 >= a.npath) return;
    const fm_edge &ed = a.ed;
    const int E = ed.E;
    constexpr int n = NL;
    unsigned char *base = smem + (size_t)wid * a.wave_bytes;
    cx<T> *cc = reinterpret_cast<cx<T> *>(base);
    T *amp = reinterpret_cast<T *>(base + a.off_amp);
    double *ang = reinterpret_cast<double *>(base + a.off_ang);
    cx<T> *cb = reinterpret_cast<cx<T> *>(base + a.off_cb);
    const int p = a.order ? a.order[a.first + s0] : a.first + s0;
    double *const rec = a.rec + (size_t)s0 * rec_len(n);
    const double R = rec[rec_len_r(n)], prod_r = rec[rec_len_r(n) + 1];
    cx<T> *const slot = reinterpret_cast<cx<T> *>(a.slot) + (size_t)s0 * slot_rows(n) * E;
    for (int e = lane; e < E; e += FM_WAVE) cc[e] = slot[e];
    wave_sync();
    // dL/dcchi: the fine grid's adjoint, or given
    double rb = 0.0;
    if (a.src.mode == 1) {
        amp_phase<T>(E, cc, amp, ang);
        rb = fine_grid_adjoint<T>(E, a.G.jq + (size_t)a.edge_id * a.nk, a.G.fq + (size_t)a.edge_id * a.nk, a.G.q,
                                  a.G.qorder, a.G.qstart + (size_t)a.edge_id * a.G.qstride, 0.5 * R * FM_BOHR,
                                  a.src.P.sigma2 ? a.src.P.sigma2[p] : 0.0,
                                  a.gseg ? a.gseg + (size_t)a.segment[p] * a.nk : nullptr, a.src.P.deg[p],
                                  a.gpath ? a.gpath + (size_t)p * a.nk : nullptr, cc, amp, ang, cb, a.nk,
                                  a.off_qs ? reinterpret_cast<double *>(base + a.off_qs) : nullptr,
                                  a.G.S ? a.G.S + (size_t)a.edge_id * a.nk * a.G.sstride : nullptr, a.G.sstride);
    } else {
        const cx<T> *gin = reinterpret_cast<const cx<T> *>(a.gcchi) + (size_t)p * E;
        for (int e = lane; e < E; e += FM_WAVE) cb[e] = gin[e];
        rb = a.greff ? a.greff[p] : 0.0;
    }
    wave_sync();
    // pbc = conj(dL/dptrac); Re(pbc D) per derivative; the cfac terms: d cfac / d r_j = a1 - a2 / r_j with
    // a1 = sum -Im(w (ck - xk)), a2 = sum Re w
    double tot[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) tot[k] = 0.0;
    for (int e = lane; e < E; e += FM_WAVE) {
        cx<T> d[NL + 3];
#pragma unroll
        for (int k = 0; k < NL + 3; ++k) d[k] = slot[(size_t)(1 + k) * E + e];
        const cx<T> cbar = cb[e];
        const cx<T> w = conj(cbar) * cc[e];
        const cx<T> wdk = w * mk<T>((T)ed.ckmxk[2 * e], (T)ed.ckmxk[2 * e + 1]);
        tot[n + 3] += (double)(-wdk.i);
        tot[n + 4] += (double)w.r;
        const cx<T> q = conj(cbar * conj(cfac_of<T>(ed, R, prod_r, e, NL)));
        slot[e] = q;
#pragma unroll
        for (int k = 0; k < NL + 3; ++k) tot[k] += (double)(q.r * d[k].r - q.i * d[k].i);
    }
    const double sum = wave_sum16(tot);
    if ((lane & 3) == 0 && (lane >> 2) < n + 5) rec[rec_sum(n) + (lane >> 2)] = sum;
    if (lane == 0) rec[rec_sum(n) + n + 5] = rb;
}

// ------------------------------------------------------------------------------------------------ the streams
constexpr int ST_MAXU = 16;
struct StreamUnit {
    double cb, sb, ch, sh, rX, rY;
    int ip, pad;
};

// Hank3T with rows 2..4 in explicit multiply-adds: which product of a two-product sum is rounded is then the same in
// every block that the seeds are used in. `last`: the last scatterer, whose 1 - z is formed from the rounded z.
template <class T> struct SeedX : Hank3T<T> {
    cx<T> rho;
    T q;
    using H = Hank3T<T>;
    __device__ __forceinline__ void init(cx<T> ck, T r) {
#pragma clang fp contract(off)
        rho = mk<T>(ck.r * r, ck.i * r);
        q = T(1) / fma(rho.r, rho.r, rho.i * rho.i);
        H::init(mk<T>(q * -rho.i, q * -rho.r), r);
    }
    // a b, the second product of the imaginary part rounded
    static __device__ __forceinline__ cx<T> mul_a(cx<T> a, cx<T> b) {
#pragma clang fp contract(off)
        return mk<T>(fma(a.r, b.r, -(a.i * b.i)), fma(a.r, b.i, a.i * b.r));
    }
    static __device__ __forceinline__ cx<T> mul_b(cx<T> a, cx<T> b) {
#pragma clang fp contract(off)
        return mk<T>(fma(a.r, b.r, -(a.i * b.i)), fma(a.i, b.r, a.r * b.i));
    }
    static __device__ __forceinline__ cx<T> fmak(cx<T> a, T k, cx<T> b) { return mk<T>(fma(a.r, k, b.r), fma(a.i, k, b.i)); }
    __device__ __forceinline__ void seeds(int r, bool last, cx<T> (&o)[3], cx<T> (&od)[3]) {
#pragma clang fp contract(off)
        const cx<T> z = this->z, zd = this->zd, zero = mk<T>(T(0), T(0)), one = mk<T>(T(1), T(0));
        const cx<T> mz = mk<T>(-z.r, -z.i), mzd = mk<T>(-zd.r, -zd.i);
        const cx<T> a = this->a1, ad = this->a1d;
        if (r == 1) {
            H::seed_row(1, o, od);
            return;
        } else if (r == 2) {
            o[0] = last ? mk<T>(T(1) - z.r, T(0) - z.i) : mk<T>(fma(q, rho.i, T(1)), fma(q, rho.r, T(0)));
            o[1] = mz;
            o[2] = od[2] = zero;
            od[0] = od[1] = mzd;
        } else if (r == 3) {
            const cx<T> v = z * T(3), zda = mul_a(zd, a), zzd = mk<T>(fma(-z.i, zd.i, z.r * zd.r), fma(z.r, zd.i, z.i * zd.r));
            o[0] = mk<T>(fma(v.i, a.i, -(v.r * a.r)) + T(1), T(0) - fma(v.r, a.i, v.i * a.r));
            od[0] = fmak(mk<T>(zda.r + fma(z.i, zd.i, -(z.r * zd.r)), zda.i + fma(z.r, -zd.i, -(z.i * zd.r))), T(-3), zero);
            o[1] = mul_b(z * T(-3), fmak(z, T(-2), one));
            od[1] = fmak(zzd, T(12), zd * T(-3));
            o[2] = mul_zz(z) * T(3);
            od[2] = zzd * T(6);
        } else {
            const cx<T> w = z * T(5), s = this->b1 + a, sd = this->b1d + ad;
            const cx<T> p = mul_a(zd, a), p2 = mul_b(z, ad), m = mul_a(w, s), g = mul_a(zd, s), g2 = mul_b(z, sd);
            o[0] = mk<T>(this->a2.r + fma(w.i, a.i, -(w.r * a.r)), this->a2.i - fma(w.r, a.i, w.i * a.r));
            od[0] = fmak(p + p2, T(-5), mzd);
            o[1] = last ? mz - m : mk<T>(fma(q, rho.i, -m.r), fma(q, rho.r, -m.i));
            od[1] = fmak(g + g2, T(-5), mzd);
            const cx<T> zz = mul_zz(z), zzd = mk<T>(fma(-z.i, zd.i, z.r * zd.r), fma(z.r, zd.i, z.i * zd.r));
            o[2] = mul_b(fmak(z, T(-3), one), zz * T(15));
            const cx<T> c = mul_b(zd, zz) * T(135);
            od[2] = fmak(zzd, T(30), mk<T>(-c.r, -c.i));
        }
        H::shift(o, od);
    }
    static __device__ __forceinline__ cx<T> mul_zz(cx<T> z) {
#pragma clang fp contract(off)
        const T h = z.r * z.i;
        return mk<T>(fma(z.r, z.r, -(z.i * z.i)), h + h);
    }
};

// The units of scatterer s (an NR x NC block) of this workgroup's paths.
template <class T, int SET, int NL, int NR, int NC>
__device__ __forceinline__ void stream_block(const MArgs<T> &a, unsigned char *smem, StreamUnit *un, double (*part)[3], int s,
                                             int row_off) {
    constexpr PairDef PD = pairdef(SET);
    constexpr KeepList KL = keep_list(SET, NR, NC);
    constexpr int NU = KL.n, NUP = (NU + 3) & ~3, RS = 2 * NUP;    // a row: the values, then their beta derivatives
    const int t = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(t / FM_WAVE), lane = lane_id();
    const fm_edge &ed = a.ed;
    const int E = ed.E, U = a.units, n = NL, ltab = ed.L1 + 1;
    const int p0 = blockIdx.x * U;
    if (t < U) {
        const int p = p0 + t < a.npath ? p0 + t : p0;
        const double *rec = a.rec + (size_t)p * rec_len(n);
        const double *tr = rec + rec_trig(n) + 4 * (s - 1);
        un[t] = StreamUnit{tr[0], tr[1], tr[2], tr[3], rec[rec_r(n) + s], rec[rec_r(n) + s - 1],
                           (int)rec[rec_pot(n) + s], 0};
    }
    __syncthreads();
    // ---- rotation tables of leg s, rows il = 2..L1 (row 1, l = 0, has constant factors and no gradient): the
    // recursion of build_tables, one (unit, representative) per lane
    for (int k0 = t; k0 < U * NU; k0 += FM_WAVE * 4) {
        const int u = k0 / NU, q = k0 - u * NU;
        int m1 = 0, m2 = 0;
#pragma unroll
        for (int r = 0; r < NU; ++r)
            if (r == q) { m1 = PD.m1[KL.k[r]]; m2 = PD.m2[KL.k[r]]; }
        const int am1 = m1 < 0 ? -m1 : m1, am2 = m2 < 0 ? -m2 : m2;
        const int mm = (m1 + 3) * 7 + (m2 + 3), nn = am1 * 4 + am2;
        const double c = un[u].cb, sn = un[u].sb, c2 = un[u].ch, s2 = un[u].sh;
        const int rows = ed.lmax1[un[u].ip];
        T *const W = reinterpret_cast<T *>(smem + (size_t)u * a.unit_bytes) + q;
        if (rows < 2) { W[0] = T(0); W[NUP] = T(0); }      // row 2 is read, with a zero t-matrix factor, by every lane
        double dlm1 = 0.0, dl = 0.0, tlm1 = 0.0, tl = 0.0;
        auto batch = [&](int il0, auto first) {
            constexpr int BATCH = 16;
            RotCoef<BATCH> rc;
            rc.fetch(ed, il0, rows, mm, nn);
#pragma unroll
            for (int v = 0; v < BATCH; ++v) {
                const int il = il0 + v;
                if (il > rows) continue;
                double d, t1;
                if (decltype(first)::value && v <= 2) {
                    d = dseed(v, m1, m2, c, sn, c2, s2);
                    t1 = dseed_db(v, m1, m2, c, sn, c2, s2);
                } else {
                    const double a1 = rc.c0[v] * c - rc.c1[v];
                    d = a1 * dl - rc.c2[v] * dlm1;
                    t1 = a1 * tl - rc.c0[v] * sn * dl - rc.c2[v] * tlm1;
                }
                dlm1 = dl; dl = d;
                tlm1 = tl; tl = t1;
                if (!(decltype(first)::value && v == 0)) {
                    W[(size_t)(il - 2) * RS] = (T)(d * rc.nr[v]);
                    W[(size_t)(il - 2) * RS + NUP] = (T)(t1 * rc.nr[v]);
                }
            }
        };
        batch(1, std::true_type{});
        for (int il0 = 17; il0 <= rows; il0 += 16) batch(il0, std::false_type{});
    }
    __syncthreads();
    // ---- the streams: lane = (unit, energy of a band of 64 / U); the bands from the highest energies (most partial
    // waves) down, dealt to the four wavefronts there and back
    const int cap = FM_WAVE / U, ul = lane / cap, il = lane % cap;
    const StreamUnit &su = un[ul];
    const int ps = p0 + ul;
    const bool valid = ps < a.npath, last = s == NL - 1;
    const T *const W0 = reinterpret_cast<const T *>(smem + (size_t)ul * a.unit_bytes);
    const T rX = (T)su.rX, rY = (T)su.rY;
    const int nb4 = (E + KB - 1) / KB, nband = (E + cap - 1) / cap;
    const T *const Kp = a.K + ((size_t)(ps / KG) * k_group(keep_rows<SET>(NL), E) + (size_t)nb4 * row_off * (KG * KB) +
                               (ps % KG) * KB) * 2;
    const T *const tl0 = TL<T>::tl(ed) + ((size_t)su.ip * ltab) * (2 * E);
    double sX = 0.0, sY = 0.0, sB = 0.0;
    for (int o = wid; o < nband; o += (o & 4) ? 2 * wid + 1 : 7 - 2 * wid) {
        const int e1 = E - o * cap, e = e1 - cap + il;          // band o: energies [e1 - cap, e1)
        const bool on = valid && e >= 0;
        const int ee = e >= 0 ? e : 0;
        cx<T> K[FM_NREP];
        {
            const T *kp = Kp + ((size_t)k_band(ee, E) * NU * (KG * KB) + k_slot(ee, E)) * 2;
#pragma unroll
            for (int q = 0; q < NU; ++q) {
                cx2<T> v;
                v.x = v.y = T(0);
                if (on) v = *reinterpret_cast<const cx2<T> *>(kp + (size_t)q * (KG * KB * 2));
                K[KL.k[q]] = mk<T>(v.x, v.y);
            }
        }
        const cx<T> pbc = reinterpret_cast<const cx<T> *>(a.slot)[(size_t)(valid ? ps : p0) * slot_rows(n) * E + ee];
        const cx<T> ck = mk<T>((T)ed.ck[2 * ee], (T)ed.ck[2 * ee + 1]);
        const int ilx = on ? ed.lmax[(size_t)su.ip * E + ee] + 1 : 1;
        const T *const tl = tl0 + 2 * ee;
        auto trow = [&](int r) {     // the t-matrix of row min(r, ilx)
            const size_t q = (size_t)(r < ilx ? r : ilx) * (2 * E);
            return mk<T>(tl[q], tl[q + 1]);
        };
        cx<T> tr = trow(2), tn = trow(3);
        cx<T> dX = mk<T>(T(0), T(0)), dY = dX, dB = dX;
        SeedX<T> X;
        Hank2T<T> Y;
        X.init(ck, rX);
        Y.init(minus_i_over(ck * rY), rY);
        cx<T> xa[3], xd[3], ya[2], yd[2];
        // rows 1..4 unrolled (their seeds are explicit per row); row 1 has constant factors and adds nothing; a lane
        // whose energy has fewer rows runs them with the t-matrix factor zero and the table's last valid row
        X.seeds(1, last, xa, xd);
        Y.seed_row(1, ya, yd);
        auto table = [&](int r, T (&w)[FM_NREP], T (&wd)[FM_NREP]) {
            const T *const w0 = W0 + (size_t)(r - 2) * RS;
#pragma unroll
            for (int q = 0; q < NU; ++q) { w[KL.k[q]] = w0[q]; wd[KL.k[q]] = w0[NUP + q]; }
        };
        T w[FM_NREP], wd[FM_NREP];
#pragma unroll
        for (int r = 2; r <= 4; ++r) {
            X.seeds(r, last, xa, xd);
            if (r < 4) Y.seed_row(r, ya, yd); else Y.step(r, ya, yd);
            const cx<T> tnn = trow(r + 2);
            const cx<T> t1 = r <= ilx ? tr : mk<T>(T(0), T(0));
            table(r <= ilx ? r : (ilx > 2 ? ilx : 2), w, wd);
            bwd_row_c<T, SET, NR, NC>(K, xa, xd, ya, yd, t1, w, wd, dX, dY, dB);
            tr = tn;
            tn = tnn;
        }
        // the row's table values read before the recursion steps that hide them, two rows per iteration so that the
        // recursions' two-row state is renamed instead of copied
        auto row = [&](int r) {
            table(r, w, wd);
            __builtin_amdgcn_sched_barrier(0);
            X.step(r, xa, xd);
            Y.step(r, ya, yd);
            const cx<T> tnn = trow(r + 2);
            bwd_row_c<T, SET, NR, NC>(K, xa, xd, ya, yd, tr, w, wd, dX, dY, dB);
            tr = tn;
            tn = tnn;
        };
        int r = 5;
#pragma unroll 1
        for (; r < ilx; r += 2) {
            row(r);
            row(r + 1);
        }
        if (r == ilx) row(r);
        if (on) {
            sX += (double)(pbc.r * dX.r - pbc.i * dX.i);
            sY += (double)(pbc.r * dY.r - pbc.i * dY.i);
            sB += (double)(pbc.r * dB.r - pbc.i * dB.i);
        }
    }
    // ---- summed over the energies: the lanes of a unit, then the wavefronts, in a fixed order
    for (int off = cap / 2; off > 0; off >>= 1) {
        sX += __shfl_xor(sX, off, FM_WAVE);
        sY += __shfl_xor(sY, off, FM_WAVE);
        sB += __shfl_xor(sB, off, FM_WAVE);
    }
    if (il == 0) {
        part[wid * ST_MAXU + ul][0] = sX;
        part[wid * ST_MAXU + ul][1] = sY;
        part[wid * ST_MAXU + ul][2] = sB;
    }
    __syncthreads();
    if (t < 3 * U && p0 + t / 3 < a.npath) {
        const int u = t / 3, k = t % 3;
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) v += part[w * ST_MAXU + u][k];
        a.rec[(size_t)(p0 + u) * rec_len(n) + rec_stream(n) + 3 * (s - 1) + k] = v;
    }
}

// Grid (ceil(npath / units), NL - 1): workgroup (b, s - 1) runs scatterer s of `units` paths.
template <class T, int SET, int NL, int WPE>
__global__ __launch_bounds__(FM_WAVE * 4) __attribute__((amdgpu_waves_per_eu(WPE))) void k_stream(MArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ StreamUnit un[ST_MAXU];
    __shared__ double part[4 * ST_MAXU][3];
    constexpr int L = lamdef(SET).L, L0 = lamdef(SET).L0;
    const int s = blockIdx.y + 1;
    if constexpr (L0 == L) {
        stream_block<T, SET, NL, L, L>(a, smem, un, part, s, keep_off<SET>(NL, s));
    } else {
        if (s == 1) stream_block<T, SET, NL, L, L0>(a, smem, un, part, s, 0);
        else if (s == NL - 1) stream_block<T, SET, NL, L0, L>(a, smem, un, part, s, keep_off<SET>(NL, s));
        else if constexpr (NL > 3) stream_block<T, SET, NL, L, L>(a, smem, un, part, s, keep_off<SET>(NL, s));
    }
}

// ------------------------------------------------------------------------------------------------ the geometry
// A workgroup of 256 threads takes as many paths as their (direction, leg) terms fit (14 of 3 legs); every term is one
// dual number through the geometry of one leg, as in the forward's regularised form.
constexpr int GE_PATHS = 14;
template <class T> __global__ __launch_bounds__(256) void k_geometry(MArgs<T> a, int per) {
    __shared__ double rat[GE_PATHS][FM_MAX_LEGS][3], gp[GE_PATHS][3 * 6], term[256];
    __shared__ int okp[GE_PATHS], pidx[GE_PATHS];
    const int t = threadIdx.x, n = a.nleg, mode = a.src.mode;
    const int q0 = blockIdx.x * per;
    if (t < per) {
        const int q = q0 + t < a.npath ? q0 + t : q0;
        const int p = a.order ? a.order[a.first + q] : a.first + q;
        int ok = 1;
        if (mode == 0) {
            for (int j = 0; j < n; ++j) {
                const int64_t ip = a.src.ipots64[(size_t)p * n + j];
                if (ip < 0 || ip >= a.src.nph1) ok = 0;
            }
        } else {
            ok = a.src.P.nleg[p] == n;
        }
        okp[t] = ok;
        pidx[t] = p;
    }
    __syncthreads();
    if (t < per * n) {
        const int q = t / n, j = t - q * n, p = pidx[q];
        double v[3];
        if (mode == 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] = a.src.coords[((size_t)p * n + j) * 3 + c] / FM_BOHR;
        } else if (okp[q]) {
            path_point(a.src.P, p, j, v);
        } else {
            v[0] = 4.0 * j; v[1] = 1.5 * (j & 1); v[2] = 0.5 * j;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) rat[q][j][c] = v[c];
    }
    // per-leg gradients: r_j (bohr) through both legs' factors, the cfac term and reff = sum r / 2; beta_j; eta_j
    if (t < per * 3 * n) {
        const int q = t / (3 * n), k = t - q * 3 * n, kind = k / n, j = k % n + 1;
        const double *rec = a.rec + (size_t)(q0 + q < a.npath ? q0 + q : q0) * rec_len(n);
        const double *sm = rec + rec_sum(n), *st = rec + rec_stream(n);
        double v;
        if (kind == 0)
            v = (j == 1 ? sm[n] : st[3 * (j - 2)]) + (j == n ? sm[n + 1] : st[3 * (j - 1) + 1]) + sm[n + 3] -
                sm[n + 4] / rec[rec_r(n) + j - 1] + 0.5 * FM_BOHR * sm[n + 5];
        else if (kind == 1)
            v = j == n ? sm[n + 2] : st[3 * (j - 1) + 2];
        else
            v = sm[j - 1];
        gp[q][k] = v;
    }
    __syncthreads();
    const int d0 = mode == 0 ? 0 : 1, ndir = 3 * (n - d0), nt = ndir * n;
    if (t < per * nt) {
        const int q = t / nt, k = t - q * nt, dir = k / n, J = k - dir * n + 1;
        const int atom = dir / 3 + d0, comp = dir % 3;
        const int i = J == n ? 0 : J, ip1 = J == n ? 1 : J + 1, im1 = J - 1;
        const int ip1a = ip1 == n ? 0 : ip1;
        double v = 0.0;
        if (atom == im1 || atom == i || atom == ip1a) {
            Dd pm[3], pi[3], pp[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pm[c] = dd(rat[q][im1][c], (im1 == atom && c == comp) ? 1.0 : 0.0);
                pi[c] = dd(rat[q][i][c], (i == atom && c == comp) ? 1.0 : 0.0);
                pp[c] = dd(rat[q][ip1a][c], (ip1a == atom && c == comp) ? 1.0 : 0.0);
            }
            const LegGeoD lg = leg_geometry_dual(pm, pi, pp);
            const int next = J == n ? 1 : J + 1;
            v = gp[q][J - 1] * lg.r.d + gp[q][n + J - 1] * lg.beta.d + gp[q][2 * n + J - 1] * lg.gamma.d +
                gp[q][2 * n + next - 1] * lg.alpha.d;
        }
        term[t] = v;
    }
    __syncthreads();
    double gout = 0.0;
    const int q = t / ndir, dir = t - q * ndir;
    const bool mine = q < per && q0 + q < a.npath;
    if (mine) {
        for (int J = 0; J < n; ++J) gout += term[q * nt + dir * n + J];
        gout = okp[q] ? gout / FM_BOHR : __builtin_nan("");
    }
    if (mode == 0) {
        if (mine) a.gcoord[(size_t)pidx[q] * a.nslot * 3 + dir] = gout;
        return;
    }
    __syncthreads();
    if (mine) {
        term[q * nt + dir] = gout;
        a.gcoord[(size_t)pidx[q] * a.nslot * 3 + 3 + dir] = gout;
    }
    __syncthreads();
    const int tail = 3 + 3 * (a.nslot - n);      // slot 0 (minus the scatterers' sum) and the unused slots
    for (int x = t; x < per * tail; x += 256) {
        const int qq = x / tail, k = x - qq * tail;
        if (q0 + qq >= a.npath) continue;
        double *out = a.gcoord + (size_t)pidx[qq] * a.nslot * 3;
        if (k < 3) {
            double s = 0.0;
            for (int j = 0; j < n - 1; ++j) s += term[qq * nt + 3 * j + k];
            out[k] = -s;
        } else {
            out[3 * n + k - 3] = 0.0;
        }
    }
}

// ------------------------------------------------------------------------------------------------ launches
constexpr size_t ST_STATIC = sizeof(StreamUnit) * ST_MAXU + sizeof(double) * 12 * ST_MAXU + 256;

template <class T, int SET, int NL> hipError_t launch_nl(const MsAdjoint &m, MArgs<T> &a, long room, const fm_launch &pol,
                                                         hipStream_t st) {
    constexpr int WPE = sizeof(T) == 4 ? 2 : 1;
    // k_chain: two wavefronts per SIMD where its matrices fit 256 registers (K edge, 3 legs: 244), else one with 512: the
    // spills cost more than the second wavefront hides (FP32, us, two / one: L3 edge, 4 legs, 38 967 paths 1988 / 1007,
    // 5 legs, 16 291 paths 1262 / 683; K edge, 4 legs, 36 909 paths 692 / 663, 5 legs, 15 111 paths 547 / 415)
    constexpr int CWPE = sizeof(T) == 4 && SET == 0 && NL <= 3 ? 2 : 1;
    constexpr int rows = keep_rows<SET>(NL);
    const fm_edge &ed = m.ed;
    const int E = ed.E;
    // k_pbc's LDS per wavefront
    size_t o = align16(sizeof(cx<T>) * E);
    a.off_amp = o; o += align16(sizeof(T) * E);
    a.off_ang = o; o += align16(sizeof(double) * E);
    a.off_cb = o; o += align16(sizeof(cx<T>) * E);
    a.off_qs = 0;
    const size_t qs = (2 * sizeof(T) + sizeof(double)) * (size_t)m.nk;
    if (m.src.mode == 1 && m.nk > 0 && sizeof(double) * 3 * (size_t)m.nk <= 32 * 1024) { a.off_qs = o; o += align16(qs); }
    a.wave_bytes = o;
    const size_t shm_c = o * 4;
    if (shm_c > FM_LDS_MAX) return hipErrorInvalidValue;
    // k_stream's LDS per unit: rows 2..L1 of the widest block
    constexpr int NUP = lamdef(SET).L0 == lamdef(SET).L || NL > 3 ? FM_NREP
                                                                  : (keep_count(SET, lamdef(SET).L, lamdef(SET).L0) + 3) & ~3;
    a.unit_bytes = path_stride(sizeof(T) * 2 * NUP * (size_t)(ed.L1 > 1 ? ed.L1 - 1 : 1));
    // the workspace: per group of 16 paths K, per path the records, the slots and, with nothing kept, the matrices
    const size_t kg = k_group(rows, E) * 2 * sizeof(T);
    const size_t b_rec = sizeof(double) * rec_len(NL), b_rt = sizeof(T) * rt_len(NL);
    const size_t b_slot = (size_t)slot_rows(NL) * E * 2 * sizeof(T);
    const size_t b_f = m.keep ? 0 : (size_t)rows * E * 2 * sizeof(T);
    const size_t group = kg + KG * (b_rec + b_rt + b_slot + b_f);
    const size_t r = (size_t)room;
    if (r < group + 2048) return hipErrorOutOfMemory;
    long chunk = (long)((r - 2048) / group) * KG;
    if (chunk > m.npath) chunk = m.npath;
    if (chunk > (1 << 23)) chunk = 1 << 23;     // k_chain: at most 4 wavefronts per path, fewer than 2^32 threads
    const size_t np = (size_t)((chunk + KG - 1) / KG) * KG;
    unsigned char *w = m.work;
    auto take = [&](size_t bytes) {
        unsigned char *p = w;
        w += (bytes + 255) & ~size_t(255);
        return p;
    };
    a.K = reinterpret_cast<T *>(take(np / KG * kg));
    a.rec = reinterpret_cast<double *>(take(np * b_rec));
    a.rt = reinterpret_cast<T *>(take(np * b_rt));
    a.slot = reinterpret_cast<T *>(take(np * b_slot));
    T *const fw = reinterpret_cast<T *>(take(np * b_f));
    const int nchunk = (E + FM_WAVE - 1) / FM_WAVE;
    if (shm_c > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)k_pbc<T, NL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm_c);
        if (e != hipSuccess) return e;
    }
    const size_t share = (WPE == 2 ? FM_LDS_SHARE : FM_LDS_MAX) - ST_STATIC;
    for (long c0 = 0; c0 < m.npath; c0 += chunk) {
        const int cnt = (int)(m.npath - c0 < chunk ? m.npath - c0 : chunk);
        a.npath = cnt;
        a.first = m.first + (int)c0;
        if (m.keep) {
            a.F = reinterpret_cast<const T *>(m.keep) + (size_t)c0 * rows * E * 2;
        } else {
            hipError_t e = forward_matrices(sizeof(T) * 8, ed, m.src, m.order, a.first, cnt, NL, fw, pol, st);
            if (e != hipSuccess) return e;
            a.F = fw;
        }
        hipLaunchKernelGGL((k_setup<T, SET>), dim3((unsigned)((cnt + 15) / 16)), dim3(256), 0, st, a);
        hipLaunchKernelGGL((k_chain<T, SET, NL, CWPE>), dim3((unsigned)(((long)cnt * nchunk + 3) / 4)), dim3(FM_WAVE * 4), 0, st, a);
        hipLaunchKernelGGL((k_pbc<T, NL>), dim3((unsigned)((cnt + 3) / 4)), dim3(FM_WAVE * 4), shm_c, st, a);
        // units per workgroup: 16 (bands of 4 energies, the most even), halved while the LDS does not hold them or the
        // launch would leave CUs without work (down to 4, whose four bands are one wavefront's each)
        int U = ST_MAXU;
        while (U > 4 && (a.unit_bytes * U > share || (long)cnt * (NL - 1) < 512L * U)) U /= 2;
        while (U > 1 && a.unit_bytes * U > FM_LDS_MAX - ST_STATIC) U /= 2;
        if (a.unit_bytes * U > FM_LDS_MAX - ST_STATIC) return hipErrorInvalidValue;
        a.units = U;
        const size_t shm_s = a.unit_bytes * U;
        if (shm_s > 48 * 1024) {
            hipError_t e = hipFuncSetAttribute((const void *)k_stream<T, SET, NL, WPE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm_s);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL((k_stream<T, SET, NL, WPE>), dim3((unsigned)((cnt + U - 1) / U), NL - 1), dim3(FM_WAVE * 4), shm_s, st, a);
        const int fit = 256 / (NL * 3 * (m.src.mode == 0 ? NL : NL - 1)), per = fit < GE_PATHS ? fit : GE_PATHS;
        hipLaunchKernelGGL(k_geometry<T>, dim3((unsigned)((cnt + per - 1) / per)), dim3(256), 0, st, a, per);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <class T> hipError_t launch_ms(const MsAdjoint &m, const fm_launch &pol, hipStream_t st) {
    MArgs<T> a;
    memset(&a, 0, sizeof a);
    a.ed = m.ed;
    a.edge_id = m.edge_id;
    a.order = m.order;
    a.src = m.src;
    a.gcchi = reinterpret_cast<const T *>(m.gcchi);
    a.greff = m.greff;
    a.G = m.G;
    a.segment = m.segment;
    a.gseg = m.gseg;
    a.gpath = reinterpret_cast<const T *>(m.gpath);
    a.gcoord = m.gcoord;
    a.nslot = m.nslot;
    a.nk = m.nk;
    a.nleg = m.nleg;
    a.once = 1;
    // the policy's paths per workgroup apply to the kernel that rebuilds the matrices; what does not fit a workgroup
    // with the rotation tables and their derivatives is refused
    const size_t lds = path_stride(align16(sizeof(PathLDS)) + 2 * align16(sizeof(T) * rot_elems(m.nleg, m.ed.L1 + 1)));
    const int g = choose_gpaths(m.ed, lds, fm_lds_budget(sizeof(T) == 4 ? 1 : 3), pol.gpaths);
    if (g == -2) return hipErrorInvalidConfiguration;
    if (g < 0) return hipErrorInvalidValue;
    const long room = (long)m.work_bytes;
    if (m.ed.ilinit <= 1) {
        switch (m.nleg) {
            case 3: return launch_nl<T, 0, 3>(m, a, room, pol, st);
            case 4: return launch_nl<T, 0, 4>(m, a, room, pol, st);
            case 5: return launch_nl<T, 0, 5>(m, a, room, pol, st);
            case 6: return launch_nl<T, 0, 6>(m, a, room, pol, st);
        }
    } else {
        switch (m.nleg) {
            case 3: return launch_nl<T, 1, 3>(m, a, room, pol, st);
            case 4: return launch_nl<T, 1, 4>(m, a, room, pol, st);
            case 5: return launch_nl<T, 1, 5>(m, a, room, pol, st);
            case 6: return launch_nl<T, 1, 6>(m, a, room, pol, st);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace

namespace fm {

size_t ms_adjoint_bytes(int precision, const fm_edge &ed, int nleg, int cnt, bool keep) {
    const size_t es = precision == 32 ? 4 : 8;
    const size_t rows = ed.ilinit <= 1 ? keep_rows<0>(nleg) : keep_rows<1>(nleg);
    const size_t path = sizeof(double) * rec_len(nleg) + es * rt_len(nleg) + slot_rows(nleg) * (size_t)ed.E * 2 * es +
                        (keep ? 0 : rows * ed.E * 2 * es);
    return (size_t)((cnt + KG - 1) / KG) * (k_group((int)rows, ed.E) * 2 * es + KG * path) + 2048;
}

size_t ms_adjoint_bytes16(int precision, int nleg) {
    const size_t ec = precision == 32 ? 8 : 16;
    const size_t rows = keep_rows<1>(nleg) > keep_rows<0>(nleg) ? keep_rows<1>(nleg) : keep_rows<0>(nleg);
    return k_group((int)rows, FM_MAX_E) * ec + KG * (sizeof(double) * (rec_len(nleg) + rt_len(nleg)) + (rows + slot_rows(nleg)) * FM_MAX_E * ec) + 4096;
}

hipError_t ms_adjoint(int precision, const MsAdjoint &a, const fm_launch &pol, hipStream_t st) {
    return precision == 32 ? launch_ms<float>(a, pol, st) : launch_ms<double>(a, pol, st);
}

}  // namespace fm
