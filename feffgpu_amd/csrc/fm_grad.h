// Per-path pieces of the adjoint kernels, one wavefront per path: the amplitude and unwrapped phase of cchi, and the
// adjoint of the fine grid (src/feffgpu/stage.py:365-388).
#pragma once
#include "fm_path.h"

namespace fm {

// Stores through a wave-uniform buffer descriptor: the lane enters as one 32-bit offset, accesses past the end write
// nothing.
constexpr int FM_RSRC_WORD3 = 0x00020000;   // buffer descriptor word 3 on gfx9: 32-bit data format, no swizzle
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rsrc(unsigned char *p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)bytes, FM_RSRC_WORD3);
}
template <class E>
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t rs, uint32_t vo, int so, const E &v) {
    if constexpr (sizeof(E) == 4) {
        unsigned x;
        __builtin_memcpy(&x, &v, 4);
        __builtin_amdgcn_raw_buffer_store_b32(x, rs, vo, so, 0);
    } else if constexpr (sizeof(E) == 8) {
        __attribute__((ext_vector_type(2))) unsigned x;
        __builtin_memcpy(&x, &v, 8);
        __builtin_amdgcn_raw_buffer_store_b64(x, rs, vo, so, 0);
    } else {
        static_assert(sizeof(E) == 16, "element of 4, 8 or 16 bytes");
        __attribute__((ext_vector_type(4))) unsigned x;
        __builtin_memcpy(&x, &v, 16);
        __builtin_amdgcn_raw_buffer_store_b128(x, rs, vo, so, 0);
    }
}

// deterministic wave sum (butterfly)
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, FM_WAVE);
    return v;
}

// amp / unwrapped phase of cc[0..E) into amp[], ang[] (the forward epilogue's first half)
template <class T>
__device__ __forceinline__ void amp_phase(int E, const cx<T> *cc, T *amp, double *ang) {
    const int lane = lane_id();
    for (int e = lane; e < E; e += FM_WAVE) {
        amp[e] = (T)sqrt((double)cc[e].r * cc[e].r + (double)cc[e].i * cc[e].i + 1e-30);
        ang[e] = (double)atan2(cc[e].i, cc[e].r);
    }
    wave_sync();
    const double a0 = ang[0];
    double dl[FM_MAX_ECHUNK];
#pragma unroll
    for (int c = 0; c < FM_MAX_ECHUNK; ++c) {
        const int e = c * FM_WAVE + lane;
        double d = 0.0;
        if (e < E && e > 0) {
            d = ang[e] - ang[e - 1];
            d -= FM_TWO_PI * rint(d / FM_TWO_PI);
        }
        dl[c] = d;
    }
    wave_sync();
    double carry = 0.0;
#pragma unroll
    for (int c = 0; c < FM_MAX_ECHUNK; ++c) {
        if (c * FM_WAVE >= E) break;
        const int e = c * FM_WAVE + lane;
        const double s = wave_scan_add(dl[c]) + carry;
        carry = __shfl(s, FM_WAVE - 1, FM_WAVE);
        if (e < E) ang[e] = a0 + s;
    }
    wave_sync();
}

// Adjoint of the fine grid of one path (one wave): chi(q) = A(q) sin(Phi(q) + 2 q reff) exp(-2 sigma2 q^2), A and
// Phi linear in amp[] and the unwrapped ang[]. From dL/dchi(q) = gup_scale gup_d[q] + gup_p[q] to dL/dcchi per
// energy: each energy gathers the q points that interpolate from it (qorder / qstart runs, in a fixed order).
// With qs (3 nk doubles of LDS), dL/dA(q), dL/dPhi(q) and the fraction are first evaluated once per q point with
// the lanes over the points (their loads independent), then gathered from LDS; without it, each energy evaluates
// them where it uses them. Returns dL/dreff (A), wave-summed.
template <class T>
__device__ __forceinline__ double fine_grid_adjoint(int E, const int32_t *jq, const double *fq, const double *q, const int32_t *qorder,
                                    const int32_t *qstart, double reff_A, double sigma2, const double *gup_d,
                                    double gup_scale, const T *gup_p, const cx<T> *cc, const T *amp, const double *ang,
                                    cx<T> *cb, int nk = 0, double *qs = nullptr, const double *S = nullptr,
                                    int sstride = 0) {
    const int lane = lane_id();
    // dL/dA and dL/dPhi at q point i from its interpolation (j, f), q and the upstream gradient gu
    auto eval = [&](int j, double f, double qi, double gu, double &gA, double &gP) {
        const double A = (1.0 - f) * (double)amp[j] + f * (double)amp[j + 1];
        double ph = (1.0 - f) * ang[j] + f * ang[j + 1] + 2.0 * qi * reff_A;
        ph -= FM_TWO_PI * rint(ph / FM_TWO_PI);
        if (sigma2 != 0.0) gu *= exp(-2.0 * sigma2 * qi * qi);
        T sn, cs;
        if constexpr (sizeof(T) == 4) sincosf((float)ph, &sn, &cs); else sincos(ph, &sn, &cs);
        gA = (double)(T)(gu * (double)sn);
        gP = (double)(T)(gu * A * (double)cs);
    };
    auto gup = [&](int i) -> double {
        double gu = 0.0;
        if (gup_d) gu += gup_scale * gup_d[i];
        if (gup_p) gu += (double)gup_p[i];
        return gu;
    };
    auto adj = [&](int i, double &gA, double &gP) { eval(jq[i], fq[i], q[i], gup(i), gA, gP); };
    double rb = 0.0;
    // dL/dcchi at energy e from dL/dA and dL/dPhi there (through amp = |cchi| and the phase)
    auto finish = [&](int e, double ab, double pb) {
        const double cr = (double)cc[e].r, ci = (double)cc[e].i;
        const double c2 = cr * cr + ci * ci, a = (double)amp[e];
        cx<T> v = mk<T>(T(0), T(0));
        if (c2 > 0.0) v = mk<T>((T)(ab * cr / a - pb * ci / c2), (T)(ab * ci / a + pb * cr / c2));
        cb[e] = v;
    };
    // staging: dL/dA and dL/dPhi per q point (values already rounded to T, so stored as T), then the fractions
    T *const sA = qs ? reinterpret_cast<T *>(qs) : nullptr;
    T *const sP = qs ? sA + nk : nullptr;
    double *const sF = qs ? reinterpret_cast<double *>(sP + nk) : nullptr;
    if (S) {   // dense interpolation (qs required): dL/dA, dL/dPhi per q point, then S^T per energy
        for (int i = lane; i < nk; i += FM_WAVE) {
            const double *Si = S + (size_t)i * sstride;
            double sa = 0.0, sp = 0.0;
            for (int e = 0; e < E; ++e) {
                sa += Si[e] * (double)amp[e];
                sp += Si[e] * ang[e];
            }
            double ph = sp + 2.0 * q[i] * reff_A;
            ph -= FM_TWO_PI * rint(ph / FM_TWO_PI);
            double gu = gup(i);
            if (sigma2 != 0.0) gu *= exp(-2.0 * sigma2 * q[i] * q[i]);
            T sn, cs;
            if constexpr (sizeof(T) == 4) sincosf((float)ph, &sn, &cs); else sincos(ph, &sn, &cs);
            const double gP = (double)(T)(gu * sa * (double)cs);
            sA[i] = (T)(gu * (double)sn);
            sP[i] = (T)gP;
            rb += 2.0 * q[i] * gP;
        }
        wave_sync();
        for (int e = lane; e < E; e += FM_WAVE) {
            double ab = 0.0, pb = 0.0;
            for (int i = 0; i < nk; ++i) {
                const double s = S[(size_t)i * sstride + e];
                ab += s * (double)sA[i];
                pb += s * (double)sP[i];
            }
            finish(e, ab, pb);
        }
        return wave_sum(rb);
    }
    if (qs) {
        const int t1 = qstart[E];
        for (int t = lane; t < t1; t += FM_WAVE) {
            const int i = qorder[t];
            double gA, gP;
            adj(i, gA, gP);
            sA[t] = (T)gA;
            sP[t] = (T)gP;
            sF[t] = fq[i];
            rb += 2.0 * q[i] * gP;
        }
        wave_sync();
        for (int e = lane; e < E; e += FM_WAVE) {
            double ab = 0.0, pb = 0.0;
            const int lo0 = qstart[e], lo1 = qstart[e + 1], hi0 = e > 0 ? qstart[e - 1] : lo0;
            for (int t = lo0; t < lo1; ++t) {
                ab += (1.0 - sF[t]) * (double)sA[t];
                pb += (1.0 - sF[t]) * (double)sP[t];
            }
            for (int t = hi0; t < lo0; ++t) {
                ab += sF[t] * (double)sA[t];
                pb += sF[t] * (double)sP[t];
            }
            finish(e, ab, pb);
        }
        return wave_sum(rb);
    }
    for (int e = lane; e < E; e += FM_WAVE) {
        double ab = 0.0, pb = 0.0;
        for (int t = qstart[e]; t < qstart[e + 1]; ++t) {    // q points with lower interpolation energy e
            const int i = qorder[t];
            double gA, gP;
            adj(i, gA, gP);
            ab += (1.0 - fq[i]) * gA;
            pb += (1.0 - fq[i]) * gP;
            rb += 2.0 * q[i] * gP;
        }
        if (e > 0)
            for (int t = qstart[e - 1]; t < qstart[e]; ++t) {  // ... and upper interpolation energy e
                const int i = qorder[t];
                double gA, gP;
                adj(i, gA, gP);
                ab += fq[i] * gA;
                pb += fq[i] * gP;
            }
        finish(e, ab, pb);
    }
    return wave_sum(rb);
}

}  // namespace fm
