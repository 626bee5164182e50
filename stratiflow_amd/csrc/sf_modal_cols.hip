// sf_modal_cols.hip -- the stage kernel of grids with few modes: one block per
// mode, one wavefront per field.
//
// A 2D grid (or a small 3D one) has fewer modes than the GPU has SIMDs, so the
// time is one wave's chain of loads, factorisations and solves and not
// bandwidth.  k_modal walks a mode's four implicit systems and its Poisson
// problem on one wavefront; here the systems of u1, u2, u3 and b run at once on
// a wavefront each while another factorises the Poisson matrix, which leaves
// one solve and the projection in the chain.  The waves exchange whole columns
// through LDS, stored [row of the lane][lane] so that lanes are consecutive.
// The arithmetic is k_modal's, operation by operation.
#include "sf_rows.h"
#include "sf_tri.h"

#include <type_traits>

namespace sf {

namespace {
// wave of each column
enum ColWave { CW_U1 = 0, CW_U3, CW_B, CW_P, CW_U2 };

template <typename T, int M>
__device__ __forceinline__ void modal_cols_body(const ModalArgs<T>& A, const int ja, const int j1,
                                                cx<T> (*const col)[M][64]) {
    using V = cx<T>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int A1 = A.A1, N = A.N3;
    const bool three = A.threeD != 0;
    const bool zero_mode = ja == 0 && j1 == 0;
    const T kx = A.kx[j1], ky = A.ky[ja], kk = A.kx2[j1], kl = A.ky2[ja];

    // this wave's column, its explicit terms of this and the previous stage
    V* x_;
    const V *n_, *ro_;
    V* rn_;
    switch (wave) {  // wave-uniform
        case CW_U1: x_ = A.u1, n_ = A.n1, ro_ = A.ro1, rn_ = A.rn1; break;
        case CW_U2: x_ = A.u2, n_ = A.n2, ro_ = A.ro2, rn_ = A.rn2; break;
        case CW_U3: x_ = A.u3, n_ = A.n3, ro_ = A.ro3, rn_ = A.rn3; break;
        case CW_B: x_ = A.b, n_ = A.nB, ro_ = A.roB, rn_ = A.rnB; break;
        default: x_ = A.p, n_ = nullptr, ro_ = nullptr, rn_ = nullptr; break;
    }
    const bool step = A.mode == 0;

    int row[M], foff[M];
#pragma unroll
    for (int t = 0; t < M; ++t) {
        row[t] = lane * M + t;
        foff[t] = row[t] < N ? int(sidx(ja, row[t], j1, N, A1) * sizeof(V)) : BUF_OOB;
    }
    const rsrc_t zr = make_rsrc(A.zl, size_t(ZC_COUNT) * M * 64 * sizeof(T));
    auto coefz = [&](int c, int t) -> T { return bld<T>(zr, lane * int(sizeof(T)), (c * M + t) * 64 * int(sizeof(T))); };
    const size_t fbytes = size_t(A1) * size_t(A.A2) * size_t(N) * sizeof(V);
    auto load = [&](const V* f, V (&g)[M]) {
        if (f == nullptr) {  // wave-uniform
#pragma unroll
            for (int t = 0; t < M; ++t) g[t] = czero<V>();
            return;
        }
        const rsrc_t r = make_rsrc(f, fbytes);
#pragma unroll
        for (int t = 0; t < M; ++t) g[t] = bld<V>(r, foff[t]);
    };
    auto store = [&](V* f, const V (&g)[M]) {
        if (f == nullptr) return;
        const rsrc_t r = make_rsrc(f, fbytes);
#pragma unroll
        for (int t = 0; t < M; ++t) bst<V>(g[t], r, foff[t]);
    };
    auto put = [&](int w, const V (&g)[M]) {
#pragma unroll
        for (int t = 0; t < M; ++t) col[w][t][lane] = g[t];
    };
    auto get = [&](int w, V (&g)[M]) {
#pragma unroll
        for (int t = 0; t < M; ++t) g[t] = col[w][t][lane];
    };
    auto zero_ends = [&](V (&g)[M], bool dir) {
#pragma unroll
        for (int t = 0; t < M; ++t) {
            const int j = row[t];
            if (j <= 1 || j >= N - 2 || (dir && j == 2)) g[t] = czero<V>();
        }
    };

    const bool solves = step && wave != CW_P;
    const bool poisson = wave == CW_P;
    const bool dir = wave == CW_U3;
    V x[M], rn[M], ro[M];
    load(x_, x);
    if (step) {
        load(n_, rn);
        load(ro_, ro);
    }
    // every coefficient this wave needs, in flight with its columns: a load
    // between two barriers would add its latency to the chain
    T dzz[3][M], z0[M], z1[M], z2[M];
    const int zlo = dir ? ZC_DZZD_LO : ZC_DZZN_LO;
    const int c0 = wave == CW_U3 ? ZC_IFULL_LO : (wave == CW_B ? ZC_S : ZC_DZDN);
#pragma unroll
    for (int t = 0; t < M; ++t) {
#pragma unroll
        for (int i = 0; i < 3; ++i) dzz[i][t] = coefz(zlo + i, t);
        z0[t] = coefz(c0, t);
        z1[t] = z2[t] = T(0);
    }
    if (dir || poisson) {
#pragma unroll
        for (int t = 0; t < M; ++t) {
            z1[t] = coefz(ZC_IFULL_DI, t);
            z2[t] = coefz(ZC_DZND, t);
        }
    }
    auto dz2 = [&](int i, int t) -> T { return dzz[i][t]; };
    const T c = wave == CW_B ? A.cb : A.cv;
    // the matrices need no field: factorised while the loads are in flight
    TriFactor<T, M> F;
    if (solves || (poisson && !(std::is_same<T, float>::value && zero_mode))) {
        T ta[M], tb[M], tc[M];
        const int kind = poisson ? 3 : (dir ? 1 : 0);
        build_rows<T, M>(kind, A, row, kk, kl, zero_mode, poisson ? T(0) : c, dz2, ta, tb, tc);
        tri_factor<T, M>(F, ta, tb, tc, lane);
    }
    if (step) {
        put(wave, x);
        sync_lds();
        if (solves) {
            V pp[M], gp[M];
            // BuildRHS linear terms (IMEXRK.cpp:140-147)
            if (!A.skip_linear) {
                if (wave == CW_U3) {
                    V bb[M], bm[M];
                    get(CW_B, bb);
                    nb_prev(bb, bm, lane);
                    if (!zero_mode) {
#pragma unroll
                        for (int t = 0; t < M; ++t) {
                            const V ifb = mad2(z0[t], bm[t], z1[t], bb[t]);
                            rn[t] = tmadc(A.Ri, ifb, rn[t]);
                        }
                    }
                } else if (wave == CW_B) {
                    V u3[M], u3p[M];
                    get(CW_U3, u3);
                    nb_next(u3, u3p, lane);
#pragma unroll
                    for (int t = 0; t < M; ++t) {
                        const V idr = cadd(cscale(T(0.5), u3[t]), cscale(T(0.5), u3p[t]));
                        rn[t] = tmadc(-z0[t], idr, rn[t]);
                    }
                }
            }
            store(rn_, rn);
            // pressure gradient
            get(CW_P, pp);
            if (wave == CW_U3) {
                V pm[M];
                nb_prev(pp, pm, lane);
#pragma unroll
                for (int t = 0; t < M; ++t) gp[t] = tscale(z2[t], csub(pp[t], pm[t]));
            } else {
                const T k = wave == CW_U1 ? kx : ky;
#pragma unroll
                for (int t = 0; t < M; ++t) gp[t] = wave == CW_B ? czero<V>() : cik(k, pp[t]);
            }
            // ExplicitRK, FinishRHS and the explicit Crank-Nicolson half
            // (IMEXRK.cpp:75-134)
            V R[M], um[M], up[M];
            nb_prev(x, um, lane);
            nb_next(x, up, lane);
#pragma unroll
            for (int t = 0; t < M; ++t) {
                const V d2 = dzz_row(dzz[0][t], um[t], dzz[1][t], x[t], dzz[2][t], up[t]);
                const V lap = cadd(mad2(kk, x[t], kl, x[t]), d2);
                R[t] = rhs_row(x[t], A.hz, ro[t], A.mh, gp[t], A.hb, rn[t], c, lap);
            }
            zero_ends(R, dir);
            tri_apply<T, M>(F, R, lane);
#pragma unroll
            for (int t = 0; t < M; ++t) x[t] = R[t];
            if (wave == CW_U1 && A.ubar != nullptr && zero_mode) {  // EvolveBackground, as in k_modal
                V ub[M];
#pragma unroll
                for (int t = 0; t < M; ++t) ub[t] = mkc<T>(row[t] < N ? A.ubar[row[t]] : T(0), T(0));
                nb_prev(ub, um, lane);
                nb_next(ub, up, lane);
#pragma unroll
                for (int t = 0; t < M; ++t) {
                    const int j = row[t];
                    const V d2 = dzz_row(dzz[0][t], um[t], dzz[1][t], ub[t], dzz[2][t], up[t]);
                    R[t] = (j <= 1 || j >= N - 2) ? czero<V>() : tmadc(A.cv, d2, ub[t]);
                }
                tri_apply<T, M>(F, R, lane);
#pragma unroll
                for (int t = 0; t < M; ++t)
                    if (row[t] < N) A.ubar[row[t]] = R[t].x;
            }
        }
        sync_lds();  // every wave has read the old columns
    }
    if (wave != CW_B) put(wave, x);
    else if (step) store(A.b, x);
    sync_lds();

    // RemoveDivergence (IMEXRK.cpp:43-73)
    if (poisson) {
        V u1[M], u2[M], u3[M], u3p[M], dv[M];
        get(CW_U1, u1);
        get(CW_U3, u3);
        if (three) get(CW_U2, u2);
        nb_next(u3, u3p, lane);
#pragma unroll
        for (int t = 0; t < M; ++t) dv[t] = div_row(kx, u1[t], three, ky, u2[t], z0[t], u3[t], u3p[t]);
        zero_ends(dv, false);
        if (std::is_same<T, float>::value && zero_mode) {
            // FP64 for the ill-conditioned pinned problem, as in k_modal; u1 and
            // u2 do not change and this wave projects u3
            T fa[M], fb[M], fc[M];
            double ta[M], tb[M], tc[M];
            build_rows<T, M>(3, A, row, kk, kl, zero_mode, T(0), dz2, fa, fb, fc);
#pragma unroll
            for (int t = 0; t < M; ++t) {
                ta[t] = fa[t];
                tb[t] = fb[t];
                tc[t] = fc[t];
            }
            TriFactor<double, M> D;
            tri_factor<double, M>(D, ta, tb, tc, lane);
            cx<double> dd[M], qm[M];
#pragma unroll
            for (int t = 0; t < M; ++t) dd[t] = mkc<double>(double(dv[t].x), double(dv[t].y));
            tri_apply<double, M>(D, dd, lane);
            nb_prev(dd, qm, lane);
#pragma unroll
            for (int t = 0; t < M; ++t) {
                const double dzq = double(z2[t]) * (dd[t].x - qm[t].x);
                const double dzqi = double(z2[t]) * (dd[t].y - qm[t].y);
                u3[t].x = T(double(u3[t].x) - dzq);
                u3[t].y = T(double(u3[t].y) - dzqi);
                x[t].x = T(double(x[t].x) + double(A.pmult) * dd[t].x);
                x[t].y = T(double(x[t].y) + double(A.pmult) * dd[t].y);
            }
            put(CW_U3, u3);
        } else {
            tri_apply<T, M>(F, dv, lane);  // dv now holds q
            put(CW_P, dv);
#pragma unroll
            for (int t = 0; t < M; ++t) x[t] = tmadc(A.pmult, dv[t], x[t]);
        }
    }
    sync_lds();
    if (wave == CW_B) return;  // no barrier below
    if (!poisson) {
        if (std::is_same<T, float>::value && zero_mode) {
            if (wave == CW_U3) get(CW_U3, x);
        } else {
            V q[M];
            get(CW_P, q);
            if (wave == CW_U3) {
                V qm[M];
                nb_prev(q, qm, lane);
#pragma unroll
                for (int t = 0; t < M; ++t) x[t] = tmadc(-z2[t], csub(q[t], qm[t]), x[t]);
            } else {
                const T k = wave == CW_U1 ? kx : ky;
#pragma unroll
                for (int t = 0; t < M; ++t) x[t] = minus_ik(k, q[t], x[t]);
            }
        }
    }
    store(x_, x);
}
}  // namespace

// threads: four waves in 2D, five in 3D
template <typename T, int M>
__global__ __launch_bounds__(320) void k_modal_cols(ModalArgs<T> A) {
    __shared__ cx<T> col[5][M][64];
    // modes of one cache line on one XCD
    const int m = xcd_tile(blockIdx.x, gridDim.x);
    modal_cols_body<T, M>(A, m / A.A1, m % A.A1, col);
}

// Up to 256 modes, or 1024 where a field is at most 1.5 MB: four or five waves
// per mode then fill the GPU in one round, and the columns, which are read a
// cache line per row, stay cheap.  Against tiles of eight modes (us per stage by
// events, tiles / columns):
//   256x1x256 FP64 (85 modes) 28.1 / 15.7      64x32x512 FP32 (399, 1.6 MB) 59.1 / 55.1
//   512x1x512 FP32 (170) 48.6 / 24.2           64x32x256 FP64 (399, 1.6 MB) 34.4 / 38.9
//   96x32x256 FP32 (608, 1.2 MB) 35.0 / 25.5   96x48x192 FP32 (992, 1.5 MB) 27.0 / 28.9
//   96x48x100 FP32 (992, 0.8 MB) 21.7 / 16.2   128x48x100 FP32 (1302, 1.0 MB) 24.4 / 31.7
// and one wave per mode for all fields, one mode per block: 21.4 us at 256x1x256
// FP64 and 8.3 us at 64x1x64 FP32, where these waves take 13.1 and 5.9 us (by
// kernel trace).
bool modal_cols_fit(int A1, int A2, int N3, int value_bytes) {
    const long modes = long(A1) * A2;
    return modes <= 256 || (modes <= 1024 && modes * N3 * value_bytes <= 1536 * 1000L);
}

template <typename T>
hipError_t launch_modal_cols(const ModalArgs<T>& a, hipStream_t s) {
    const dim3 grid(a.A1 * a.A2), block(a.threeD ? 320 : 256);
    switch ((a.N3 + 63) / 64) {
#define SF_M(m)                                                            \
    case m:                                                                \
        hipLaunchKernelGGL((k_modal_cols<T, m>), grid, block, 0, s, a);    \
        break;
        SF_M(1) SF_M(2) SF_M(3) SF_M(4) SF_M(5) SF_M(6) SF_M(7) SF_M(8)
#undef SF_M
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template hipError_t launch_modal_cols<float>(const ModalArgs<float>&, hipStream_t);
template hipError_t launch_modal_cols<double>(const ModalArgs<double>&, hipStream_t);

}  // namespace sf
