// sf_rows.h -- a mode's column on one wavefront: neighbouring rows and the rows
// of its vertical systems.
#pragma once
#include "sf_kernels.h"
#include "sf_tri.h"

namespace sf {

// the rows before and after each row of the lane
template <int M, typename V>
__device__ __forceinline__ void nb_prev(const V (&x)[M], V (&xm)[M], int lane) {
    V s = shfl_idx(x[M - 1], (lane - 1) & 63);
    if (lane == 0) s = czero<V>();
    xm[0] = s;
#pragma unroll
    for (int t = 1; t < M; ++t) xm[t] = x[t - 1];
}
template <int M, typename V>
__device__ __forceinline__ void nb_next(const V (&x)[M], V (&xp)[M], int lane) {
    V s = shfl_idx(x[0], (lane + 1) & 63);
    if (lane == 63) s = czero<V>();
#pragma unroll
    for (int t = 0; t < M - 1; ++t) xp[t] = x[t + 1];
    xp[M - 1] = s;
}

// a*x + b*y with the roundings of fma(a, x, b*y)
template <typename V, typename T>
__device__ __forceinline__ V mad2(T a, V x, T b, V y) {
    return tmadc(a, x, tscale(b, y));
}
// second difference lo*um + di*u + up*un of a column's row
template <typename V, typename T>
__device__ __forceinline__ V dzz_row(T lo, V um, T di, V u, T up, V un) {
    return tmadc(up, un, mad2(lo, um, di, u));
}
// divergence ikx u1 + iky u2 + dzdn (u3' - u3), u2 not read in 2D
template <typename V, typename T>
__device__ __forceinline__ V div_row(T kx, V u1, bool three, T ky, V u2, T dzdn, V u3, V u3p) {
    V h = mkc<T>(tmul(-kx, u1.y), tmul(kx, u1.x));
    if (three) h = mkc<T>(tmad(-kx, u1.y, tmul(-ky, u2.y)), tmad(kx, u1.x, tmul(ky, u2.x)));
    return tmadc(dzdn, csub(u3p, u3), h);
}

// u - ik q
template <typename V, typename T>
__device__ __forceinline__ V minus_ik(T k, V q, V u) {
    return mkc<T>(tmad(k, q.y, u.x), tmad(-k, q.x, u.y));
}
// explicit right-hand side u + hz ro + mh grad p + hb rn + c Lap u of a row
template <typename V, typename T>
__device__ __forceinline__ V rhs_row(V u, T hz, V ro, T mh, V gp, T hb, V rn, T c, V lap) {
    return tmadc(c, lap, tmadc(hb, rn, tmadc(mh, gp, tmadc(hz, ro, u))));
}

// kind: 0 velocity Neumann, 1 velocity Dirichlet, 2 buoyancy Neumann,
// 3 pressure Laplacian.  Matrix rows as built in IMEXRK.h:55-78, 502-545
// with Neumannify/Dirichlify (Differentiation.h:17-59).
// zcoef(i, t): sub-, main and super-diagonal (i = 0, 1, 2) of the second
// derivative at the lane's row t (zero beyond N3), Dirichlet for kind 1, else
// Neumann.
template <typename T, int M, typename ZC>
__device__ __forceinline__ void build_rows(int kind, const ModalArgs<T>& A, const int (&row)[M], T kk, T kl,
                                           bool zero_mode, T coef, ZC zcoef, T (&a)[M], T (&b)[M], T (&c)[M]) {
    const int N = A.N3;
    const bool dir = (kind == 1);
#pragma unroll
    for (int t = 0; t < M; ++t) {
        const int j = row[t];
        if (j >= N) {
            a[t] = 0;
            b[t] = 1;
            c[t] = 0;
            continue;
        }
        const T lo = zcoef(0, t), di = zcoef(1, t), up = zcoef(2, t);
        const T ldi = (di + kk) + kl;
        T aa, bb, cc;
        if (kind == 3) {
            aa = lo;
            bb = ldi;
            cc = up;
        } else {
            aa = -(coef * lo);
            bb = T(1) - coef * ldi;
            cc = -(coef * up);
        }
        if (j == 0) aa = 0;
        if (j == N - 1) cc = 0;
        if (!dir) {
            if (j == 0) {
                bb = 1;
                cc = 0;
            } else if (j == 1) {
                aa = 0;
                bb = 1;
                cc = -1;
            } else if (j == N - 2) {
                aa = 1;
                bb = -1;
                cc = 0;
            } else if (j == N - 1) {
                aa = 0;
                bb = 1;
            }
        } else if (j <= 2 || j >= N - 2) {
            aa = 0;
            bb = 1;
            cc = 0;
        }
        if (kind == 3 && zero_mode && j <= 1) {
            aa = 0;
            bb = 1;
            cc = 0;
        }
        a[t] = aa;
        b[t] = bb;
        c[t] = cc;
    }
}

}  // namespace sf
