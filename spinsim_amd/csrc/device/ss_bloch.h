// Bloch vector of one state (get_spin, spinsim/__init__.py:936-944), shared by
// the GPU scans, the GPU spin kernel and the host (CPU device) build.
#pragma once

// Written with explicit fused multiply-adds on the GPU, so that every kernel that
// stores a state's vector stores the same bits.
#ifdef SS_HOST
#define SS_BLOCH_FMA(a, b, c) ((a) * (b) + (c))
#else
#define SS_BLOCH_FMA(a, b, c) fma(a, b, c)
#endif

template <int D>
static __device__ __forceinline__ void ss_store_spin(const ss_cd s[D], double* spin, long long i)
{
    double sx, sy, sz;
    if (D == 2) {
        // Re and -Im of psi0 psi1*, and (|psi0|^2 - |psi1|^2) / 2
        sx = SS_BLOCH_FMA(s[0].x, s[1].x, s[0].y * s[1].y);
        sy = SS_BLOCH_FMA(s[0].x, s[1].y, -(s[0].y * s[1].x));
        sz = 0.5 * SS_BLOCH_FMA(s[0].x, s[0].x,
                                SS_BLOCH_FMA(s[0].y, s[0].y, SS_BLOCH_FMA(-s[1].x, s[1].x, -(s[1].y * s[1].y))));
    } else {
        const double r2 = 1.4142135623730951;
        const ss_cd u = ss_add(s[0], s[D - 1]);
        const ss_cd v = ss_c(s[0].x - s[D - 1].x, s[0].y - s[D - 1].y);
        // sqrt2 Re(psi1* u), -sqrt2 Im(psi1* v), |psi0|^2 - |psi2|^2
        sx = r2 * SS_BLOCH_FMA(s[1].x, u.x, s[1].y * u.y);
        sy = -r2 * SS_BLOCH_FMA(s[1].x, v.y, -(s[1].y * v.x));
        sz = SS_BLOCH_FMA(s[0].x, s[0].x, SS_BLOCH_FMA(s[0].y, s[0].y,
                          SS_BLOCH_FMA(-s[D - 1].x, s[D - 1].x, -(s[D - 1].y * s[D - 1].y))));
    }
    spin[3 * i + 0] = sx;
    spin[3 * i + 1] = sy;
    spin[3 * i + 2] = sz;
}
