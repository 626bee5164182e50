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

// PROJECT: the projection alone, in a kernel of its own for FP64: with the registers
// of a stage, columns of more than 320 levels spill up to 182 of them (projection
// of 256x1x512: 19.8 us in the stage's kernel, 12.7 in its own; 256x1x384: 12.8 and
// 10.5).  In FP32 the kernel of its own is no faster, its registers are those of the
// (0,0) mode's FP64 solve (96x32x100: 6.1 us in the stage's kernel, 7.4 in its own).
// A stage asks the mode at run time: fixed at compile time its allocation spills
// more at 384 levels (256x1x384 FP64: 21.1 -> 24.5 us).
template <typename T, int M, bool PROJECT>
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

    const bool step = !PROJECT && A.mode == 0;

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
template <typename T, int M, bool PROJECT>
__global__ __launch_bounds__(320) void k_modal_cols(ModalArgs<T> A) {
    __shared__ cx<T> col[5][M][64];
    // modes of one cache line on one XCD
    const int m = xcd_tile(blockIdx.x, gridDim.x);
    modal_cols_body<T, M, PROJECT>(A, m / A.A1, m % A.A1, col);
}

// Up to one mode per CU the columns are the faster kernel by far (us per stage by
// events, tiles of eight modes / columns: 256x1x256 FP64, 85 modes, 28.5 / 15.4;
// 512x1x512 FP32, 170 modes, 35.8 / 21.0; one wave per mode for all fields took
// 21.4 us at 256x1x256 FP64 where these take 13.1 by kernel trace).  With more modes a
// CU runs two, three or four blocks at once, which compete for its LDS and
// registers the more the longer the columns are, and tiles read whole cache lines
// where columns read a value of a line each.  Rows of whole groups of eight modes
// keep the modes of a line on one XCD (xcd_tile needs their number to divide by
// eight), ragged rows do not and reach the crossover earlier; of rows of two
// modes a tile uses only two of its eight places.  Stage, tiles / columns:
//   2 modes per CU, whole              48x48x512 FP32 45.1 / 34.1   48x48x384 FP64 47.0 / 40.3, x512 77.2 / 82.3
//              2, ragged              64x32x256 FP32 31.9 / 23.8, x384 36.9 / 39.0    x192 FP64 37.8 / 32.8, x256 36.0 / 38.7
//              3, whole               96x32x256 FP32 30.3 / 23.3, x384 35.9 / 37.7    x192 FP64 35.9 / 29.9, x256 33.0 / 34.7
//              3, ragged              64x48x128 FP32 23.0 / 20.8, x192 26.4 / 32.1    x100 FP64 30.7 / 28.2, x128 31.8 / 33.1
//              4, whole               96x48x128 FP32 22.5 / 17.4, x192 25.9 / 27.3    x128 FP64 30.5 / 28.7, x192 37.5 / 39.5
//              4, ragged              64x64x100 FP32 23.4 / 22.0, x128 23.6 / 26.7    x64 FP64 25.7 / 22.0, x100 31.6 / 37.9
// (128x48x64, 1302 modes: FP32 19.9 / 21.4, FP64 26.7 / 30.1.)  The projection alone has
// one solve to spread over the waves and crosses over at shorter columns: whole
// 48x48x256 FP32 10.5 / 8.9, x384 12.7 / 14.4, x192 FP64 9.9 / 8.5, x384 15.5 / 17.3;
// 96x48x192 FP32 9.8 / 14.5, x100 FP64 8.7 / 10.2; ragged 64x48x100 FP32 8.4 / 10.2.
bool modal_cols_fit(int A1, int A2, int N3, int value_bytes, bool step) {
    // levels up to which the columns are taken, by modes per CU (2, 3, 4)
    static const int levels[2][2][2][3] = {
        {{{0, 0, 0}, {0, 0, 0}}, {{256, 100, 48}, {192, 128, 64}}},              // projection: ragged, whole; FP32, FP64
        {{{256, 128, 100}, {192, 100, 64}}, {{512, 256, 128}, {384, 192, 128}}}  // step
    };
    const long modes = long(A1) * A2;
    if (modes <= 256) return true;
    if (modes > 1024) return false;
    const bool whole = A1 % 8 == 0 || A1 < 4;
    const int per_cu = A1 < 4 ? 2 : int((modes + 255) / 256);
    return N3 <= levels[step][whole][value_bytes == 16][per_cu - 2];
}

template <typename T>
hipError_t launch_modal_cols(const ModalArgs<T>& a, hipStream_t s) {
    const dim3 grid(a.A1 * a.A2), block(a.threeD ? 320 : 256);
    switch ((a.N3 + 63) / 64) {
#define SF_M(m)                                                                        \
    case m:                                                                            \
        if constexpr (std::is_same<T, double>::value) {                                \
            if (a.mode != 0) {                                                         \
                hipLaunchKernelGGL((k_modal_cols<T, m, true>), grid, block, 0, s, a);  \
                break;                                                                 \
            }                                                                          \
        }                                                                              \
        hipLaunchKernelGGL((k_modal_cols<T, m, false>), grid, block, 0, s, a);         \
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
