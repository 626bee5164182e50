// sf_precond.hip -- the advected diffusion preconditioner (its diffusion-only
// form, a real system, is k_diffprec in sf_kernels_impl.h).
#include "sf_kernels.h"

#include <type_traits>

namespace sf {

namespace {
template <typename V>
__device__ __forceinline__ V shfl_c(V v, int src) {
    V r;
    r.x = __shfl(v.x, src, 64);
    r.y = __shfl(v.y, src, 64);
    return r;
}
template <typename V>
__device__ __forceinline__ V crecip(V a) {
    const auto r = decltype(a.x)(1) / (a.x * a.x + a.y * a.y);
    V o;
    o.x = r * a.x;
    o.y = -r * a.y;
    return o;
}

// Solves one complex tridiagonal system per wavefront in place: lane l owns
// rows l*M .. l*M+M-1 with real off-diagonals a, c (a[0] of lane 0 and c[M-1]
// of lane 63 zero; padding rows identity), complex diagonal b and right-hand
// side d.  The scheme of sf_tri.h with complex factors and one right-hand side:
// each lane eliminates its M-1 interior rows (g, spikes v and w), the 64
// interface rows form a Schur system solved by parallel cyclic reduction.
template <typename T, int M>
__device__ __forceinline__ void ctri_solve(const T (&a)[M], const cx<T> (&b)[M], const T (&c)[M], cx<T> (&d)[M],
                                           int lane) {
    using V = cx<T>;
    V As, Bs, Cs, Ds;
    V g[M], v[M], w[M];
    if constexpr (M == 1) {
        As = mkc<T>(a[0], 0);
        Bs = b[0];
        Cs = mkc<T>(c[0], 0);
        Ds = d[0];
    } else {
        V r[M], cc[M];
        r[0] = crecip(b[0]);
#pragma unroll
        for (int t = 0; t < M - 2; ++t) {
            cc[t] = cscale(c[t], r[t]);
            r[t + 1] = crecip(csub(b[t + 1], cscale(a[t + 1], cc[t])));
        }
        g[0] = cmul(r[0], d[0]);
        v[0] = cscale(a[0], r[0]);
#pragma unroll
        for (int t = 1; t <= M - 2; ++t) {
            g[t] = cmul(r[t], csub(d[t], cscale(a[t], g[t - 1])));
            v[t] = cmul(r[t], cscale(-a[t], v[t - 1]));
        }
        w[M - 2] = cscale(c[M - 2], r[M - 2]);
#pragma unroll
        for (int t = M - 3; t >= 0; --t) {
            g[t] = csub(g[t], cmul(cc[t], g[t + 1]));
            v[t] = csub(v[t], cmul(cc[t], v[t + 1]));
            w[t] = cscale(T(-1), cmul(cc[t], w[t + 1]));
        }
        V gn = shfl_c(g[0], (lane + 1) & 63), vn = shfl_c(v[0], (lane + 1) & 63), wn = shfl_c(w[0], (lane + 1) & 63);
        if (lane == 63) gn = vn = wn = czero<V>();
        const T aI = a[M - 1], cI = c[M - 1];
        As = cscale(-aI, v[M - 2]);
        Bs = csub(csub(b[M - 1], cscale(aI, w[M - 2])), cscale(cI, vn));
        Cs = cscale(-cI, wn);
        Ds = csub(csub(d[M - 1], cscale(aI, g[M - 2])), cscale(cI, gn));
    }
#pragma unroll
    for (int lev = 0; lev < 6; ++lev) {
        const int s = 1 << lev;
        const int lo = (lane - s) & 63, hi = (lane + s) & 63;
        V Am = shfl_c(As, lo), Bm = shfl_c(Bs, lo), Cm = shfl_c(Cs, lo), Dm = shfl_c(Ds, lo);
        V Ap = shfl_c(As, hi), Bp = shfl_c(Bs, hi), Cp = shfl_c(Cs, hi), Dp = shfl_c(Ds, hi);
        if (lane - s < 0) {
            Am = Cm = Dm = czero<V>();
            Bm = mkc<T>(1, 0);
        }
        if (lane + s > 63) {
            Ap = Cp = Dp = czero<V>();
            Bp = mkc<T>(1, 0);
        }
        const V al = cscale(T(-1), cmul(As, crecip(Bm)));
        const V ga = cscale(T(-1), cmul(Cs, crecip(Bp)));
        Bs = cadd(Bs, cadd(cmul(al, Cm), cmul(ga, Ap)));
        Ds = cadd(Ds, cadd(cmul(al, Dm), cmul(ga, Dp)));
        As = cmul(al, Am);
        Cs = cmul(ga, Cp);
    }
    const V sl = cmul(Ds, crecip(Bs));
    if constexpr (M > 1) {
        V sm = shfl_c(sl, (lane - 1) & 63);
        if (lane == 0) sm = czero<V>();
#pragma unroll
        for (int t = 0; t <= M - 2; ++t) d[t] = csub(csub(g[t], cmul(v[t], sm)), cmul(w[t], sl));
    }
    d[M - 1] = sl;
}
}  // namespace

// out = (tnu (Dzz - k^2) - i tadv kx U(z) - delta)^-1 ZeroEnds(in) - in/2 on
// the modes with |k|^2 <= k2max, -in on the others; solved as
//   (I - coef (Dzz - k^2) + i adv U) x = -ZeroEnds(in)/delta,
// coef = tnu/delta, adv = tadv kx/delta: strictly diagonally dominant for
// delta > 0 but for the Neumannified rows.
//
// FP64: one wavefront per mode, MB modes of consecutive j1 per block.  A sweep down
// the column on one lane per mode is a chain of N3 dependent divisions and
// global loads in each direction (182 us for a 256x1x256 FP64 field whatever
// its number of modes); here the chain is M - 1 rows and six exchanges long.
// Few modes (a 2D grid): one mode per block, its column read directly, so
// that every mode has a CU of its own; else eight, staged through an LDS tile
// so that HBM sees runs of eight modes.
template <typename T, int M, int MB>
__global__ __launch_bounds__(MB * 64) void k_advprec(DiffPrecArgs<T> P) {
    using V = cx<T>;
    constexpr int TP = MB + 1;
    __shared__ V tile[MB > 1 ? 64 * M * TP : 1];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int N = P.N3, A1 = P.A1;
    const int ja = blockIdx.y, j10 = blockIdx.x * MB;
    const int j1 = min(j10 + wave, A1 - 1);  // waves past A1 solve a mode again and store nothing
    const int cw = int(threadIdx.x) % MB, cz = int(threadIdx.x) / MB;
    V x[M];
    if constexpr (MB > 1) {
        for (int z = cz; z < 64 * M; z += 64)
            tile[z * TP + cw] = (z < N && j10 + cw < A1) ? P.in[sidx(ja, z, j10 + cw, N, A1)] : czero<V>();
        __syncthreads();
#pragma unroll
        for (int t = 0; t < M; ++t) x[t] = tile[(lane * M + t) * TP + wave];
    } else {
#pragma unroll
        for (int t = 0; t < M; ++t) x[t] = lane * M + t < N ? P.in[sidx(ja, lane * M + t, j1, N, A1)] : czero<V>();
    }
    const T kk = P.kx2[j1], kl = P.ky2[ja];
    V y[M];
    if (-(kk + kl) <= P.k2max) {  // wave-uniform
        const bool dir = P.dirichlet != 0;
        const T coef = P.tnu / P.delta, rs = T(-1) / P.delta, adv = P.tadv * P.kx[j1] / P.delta;
        const T* lo = P.zc + (dir ? ZC_DZZD_LO : ZC_DZZN_LO) * P.N3p;
        const T* ub = P.zc + ZC_UBAR * P.N3p;
        T a[M], c[M];
        V b[M];
#pragma unroll
        for (int t = 0; t < M; ++t) {
            const int j = lane * M + t;
            const int jc = min(j, N - 1);
            a[t] = -(coef * lo[jc]);
            b[t].x = T(1) - coef * ((lo[P.N3p + jc] + kk) + kl);
            b[t].y = adv * ub[jc];
            c[t] = -(coef * lo[2 * P.N3p + jc]);
            const bool end = j <= 1 || j >= N - 2 || (dir && j == 2);
            y[t] = end ? czero<V>() : cscale(rs, x[t]);
            // rows with the Neumannify/Dirichletify replacements of the
            // implicit solves; identity beyond the column
            const bool ident = dir ? end : (j == 0 || j >= N - 1);
            if (ident) {
                a[t] = c[t] = 0;
                b[t] = mkc<T>(1, 0);
            } else if (!dir && j == 1) {
                a[t] = 0;
                b[t] = mkc<T>(1, 0);
                c[t] = -1;
            } else if (!dir && j == N - 2) {
                a[t] = 1;
                b[t] = mkc<T>(-1, 0);
                c[t] = 0;
            }
        }
        ctri_solve<T, M>(a, b, c, y, lane);
#pragma unroll
        for (int t = 0; t < M; ++t) y[t] = csub(y[t], cscale(T(0.5), x[t]));
    } else {
#pragma unroll
        for (int t = 0; t < M; ++t) y[t] = cscale(T(-1), x[t]);
    }
    if constexpr (MB > 1) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < M; ++t) tile[(lane * M + t) * TP + wave] = y[t];
        __syncthreads();
        for (int z = cz; z < N; z += 64)
            if (j10 + cw < A1) P.out[sidx(ja, z, j10 + cw, N, A1)] = tile[z * TP + cw];
    } else {
#pragma unroll
        for (int t = 0; t < M; ++t)
            if (lane * M + t < N) P.out[sidx(ja, lane * M + t, j1, N, A1)] = y[t];
    }
}

// FP32: a Thomas sweep per mode on one lane, which keeps the rounding of every
// operation in its place (results of the wavefront form differ by 1e-7).  Its
// chain is a complex division per row; what it needs from memory does not have
// to be in that chain: the block stages its SWEEP_T columns and the
// coefficient rows in LDS first and writes the result back at the end.
constexpr int SWEEP_T = 8;  // modes per block: N3 = 512 takes 72 KB of LDS
constexpr int SWEEP_BS = 64;
template <typename T>
__global__ __launch_bounds__(SWEEP_BS) void k_advprec_sweep(DiffPrecArgs<T> P) {
    using V = cx<T>;
    extern __shared__ unsigned char adv_lds[];
    const int N = P.N3;
    V* cp = reinterpret_cast<V*>(adv_lds);  // [z][SWEEP_T]: modified super-diagonal
    V* dp = cp + N * SWEEP_T;               // [z][SWEEP_T]: input, then modified right-hand side
    T* zl = reinterpret_cast<T*>(dp + N * SWEEP_T);  // sub-, main and super-diagonal of Dzz, U
    const bool dir = P.dirichlet != 0;
    const int lo = dir ? ZC_DZZD_LO : ZC_DZZN_LO;
    const int ja = blockIdx.y, j10 = blockIdx.x * SWEEP_T;
    for (int i = threadIdx.x; i < N * SWEEP_T; i += SWEEP_BS) {
        const int z = i / SWEEP_T, j1 = j10 + i % SWEEP_T;
        dp[i] = j1 < P.A1 ? P.in[sidx(ja, z, j1, N, P.A1)] : czero<V>();
    }
    for (int z = threadIdx.x; z < N; z += SWEEP_BS) {
#pragma unroll
        for (int c = 0; c < 3; ++c) zl[c * N + z] = P.zc[(lo + c) * P.N3p + z];
        zl[3 * N + z] = P.zc[ZC_UBAR * P.N3p + z];
    }
    __syncthreads();
    const int t = threadIdx.x;
    const int j1 = min(j10 + t, P.A1 - 1);
    const T kk = P.kx2[j1], kl = P.ky2[ja];
    if (t < SWEEP_T && !(-(kk + kl) > P.k2max)) {
        const T coef = P.tnu / P.delta;
        const T rs = T(-1) / P.delta;
        const T adv = P.tadv * P.kx[j1] / P.delta;
        // rows of (I - coef (Dzz - k^2) + i adv U) with the Neumannify/Dirichletify
        // replacements of the implicit solves
        auto rowc = [&](int j, T& a, V& b, T& c) {
            a = -(coef * zl[j]);
            b.x = T(1) - coef * ((zl[N + j] + kk) + kl);
            b.y = adv * zl[3 * N + j];
            c = -(coef * zl[2 * N + j]);
            if (j == 0) a = 0;
            if (j == N - 1) c = 0;
            const bool id = dir ? (j <= 2 || j >= N - 2) : (j == 0 || j == N - 1);
            if (id) {
                a = 0;
                b = mkc<T>(1, 0);
                c = 0;
            } else if (!dir && j == 1) {
                a = 0;
                b = mkc<T>(1, 0);
                c = -1;
            } else if (!dir && j == N - 2) {
                a = 1;
                b = mkc<T>(-1, 0);
                c = 0;
            }
        };
        auto rhs = [&](int j) {
            const bool end = j <= 1 || j >= N - 2 || (dir && j == 2);
            return end ? czero<V>() : cscale(rs, dp[j * SWEEP_T + t]);
        };
        auto cdiv = [](V a, V b) {
            const T r = T(1) / (b.x * b.x + b.y * b.y);
            return cscale(r, cmulc(a, b));
        };
        V cprev = czero<V>(), dprev = czero<V>();
#pragma unroll 4
        for (int j = 0; j < N; ++j) {
            T a, c;
            V b;
            rowc(j, a, b, c);
            const V den = csub(b, cscale(a, cprev));
            const V cj = cdiv(mkc<T>(c, 0), den);
            const V dj = cdiv(csub(rhs(j), cscale(a, dprev)), den);
            cp[j * SWEEP_T + t] = cj;
            dp[j * SWEEP_T + t] = dj;
            cprev = cj;
            dprev = dj;
        }
        V x = dprev;
#pragma unroll 4
        for (int j = N - 2; j >= 0; --j) {
            x = csub(dp[j * SWEEP_T + t], cmul(cp[j * SWEEP_T + t], x));
            dp[j * SWEEP_T + t] = x;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < N * SWEEP_T; i += SWEEP_BS) {
        const int z = i / SWEEP_T, j1 = j10 + i % SWEEP_T;
        if (j1 >= P.A1) continue;
        const size_t e = sidx(ja, z, j1, N, P.A1);
        P.out[e] = -(P.kx2[j1] + kl) > P.k2max ? cscale(T(-1), P.in[e]) : csub(dp[i], cscale(T(0.5), P.in[e]));
    }
}

template <typename T, int M>
static void launch_advprec_m(const DiffPrecArgs<T>& p, hipStream_t s) {
    // up to four modes per CU the GPU is not filled by one mode per block
    if (p.A1 * p.A2 <= 1024)
        hipLaunchKernelGGL((k_advprec<T, M, 1>), dim3(p.A1, p.A2), dim3(64), 0, s, p);
    else
        hipLaunchKernelGGL((k_advprec<T, M, 8>), dim3((p.A1 + 7) / 8, p.A2), dim3(512), 0, s, p);
}

template <typename T>
hipError_t launch_advprec(const DiffPrecArgs<T>& p, hipStream_t s) {
    if (p.A1 <= 0 || p.A2 <= 0 || p.in == p.out || !(p.delta > T(0)) || p.N3 > advprec_rows<T>())
        return hipErrorInvalidValue;
    if constexpr (std::is_same<T, float>::value) {
        const size_t lds = size_t(p.N3) * (2 * SWEEP_T * sizeof(cx<T>) + 4 * sizeof(T));
        if (lds > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_advprec_sweep<T>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL((k_advprec_sweep<T>), dim3((p.A1 + SWEEP_T - 1) / SWEEP_T, p.A2), dim3(SWEEP_BS), lds, s, p);
    } else {
        static_assert(advprec_rows<double>() == 256, "up to four rows per lane");
        switch ((p.N3 + 63) / 64) {
            case 1: launch_advprec_m<T, 1>(p, s); break;
            case 2: launch_advprec_m<T, 2>(p, s); break;
            case 3: launch_advprec_m<T, 3>(p, s); break;
            case 4: launch_advprec_m<T, 4>(p, s); break;
            default: return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

template hipError_t launch_advprec<float>(const DiffPrecArgs<float>&, hipStream_t);
template hipError_t launch_advprec<double>(const DiffPrecArgs<double>&, hipStream_t);

}  // namespace sf
