// sf_transform.hip -- x transforms of whole fields between the nodal layout
// (z fastest) and the x-spectral layout (x mode fastest): ToNodal, ToModal,
// PopulateNodalVariables, the CFL number and the adjoint step.
#include "sf_fft.h"
#include "sf_kernels.h"

namespace sf {

namespace {
constexpr int BS = 256;

// A real line of N1 points is a complex FFT of N1/2: even points in the real
// and odd points in the imaginary part, one multiplication by w^k = exp(-2 pi i
// k/N1) per mode before (inverse) or after it (forward).  Half the work of a
// complex line per level, and each level's result depends on that level alone
// (two levels in one line would round equal levels differently).
//
// NL levels per block: 16, or 8 where the lines are long.  Their LDS (26 KB at
// 384 points in FP32) leaves room for six blocks per CU, whose loads, FFTs and
// stores overlap; the nodal side moves runs of NL levels (64 bytes).
template <typename T, int N1>
constexpr int xt_levels() {
    return N1 * int(sizeof(cx<T>)) > 4096 ? 8 : 16;
}

// FFT plan of a line of M points.  A block has 16 lines of 24 or 32 points
// (N1 = 48 and 64): one DFT per lane would leave 240 of its 256 threads idle
// through the longest chain of the kernel, two passes use 96 or 128 of them.
template <int M>
constexpr int xt_plan() {
    return M == 24 || M == 32 ? 4 : 0;
}

// line pitch of 2 mod 16 complex values: the lanes that touch one point of the
// block's lines for the nodal side fall into distinct LDS banks
template <int M>
constexpr int xt_ldp() {
    using P = FftPlan<M, xt_plan<M>()>;
    int l = P::two ? M + P::R2 : M;
    while (l % 16 != 2) ++l;
    return l;
}
}  // namespace

template <typename T, int N1>
__global__ __launch_bounds__(BS) void k_x_c2r(XTArgs<T> A) {
    using V = cx<T>;
    constexpr int M = N1 / 2, LDP = xt_ldp<M>(), NL = xt_levels<T, N1>();
    __shared__ V buf[NL * LDP];
    const int N3 = A.N3, A1 = A.A1;
    // z blocks of one n2, which share the nodal side's cache lines, on one XCD;
    // where every block writes whole lines the blocks keep their order, since an
    // XCD for every few planes only puts the XCDs a power of two apart (ToNodal
    // of 128x128x128 FP64 19.7 -> 15.0 us, 192x96x192 FP64 27.2 -> 24.3)
    constexpr int LINE = 128 / int(sizeof(T));
    const int block = blockIdx.x + gridDim.x * blockIdx.y;
    const int tile = NL % LINE == 0 && N3 % LINE == 0 ? block : xcd_tile(block, gridDim.x * gridDim.y);
    const int n2 = tile / gridDim.x, z0 = (tile % gridDim.x) * NL;
    const V* __restrict__ in = A.spec[blockIdx.z];
    T* __restrict__ out = A.nodal[blockIdx.z];
    const V* __restrict__ wt = A.tw + 2 * M;
    const bool dx = (A.ikx >> blockIdx.z) & 1;
    // modes k and M - k of a level give points k and M - k of its line:
    //   Z_k = (X_k + conj X_{M-k}) + i conj(w^k) (X_k - conj X_{M-k})
    constexpr int H = M / 2 + 1;
    for (int idx = threadIdx.x; idx < NL * H; idx += BS) {
        const int t = idx / H;
        const int k = idx - t * H;
        const int z = z0 + t;
        V a = czero<V>(), b = czero<V>();
        if (z < N3) {
            const V* X = in + sidx(n2, z, 0, N3, A1);
            if (k < A1) a = X[k];
            if (M - k < A1) b = X[M - k];
        }
        if (dx) {  // ikx X
            a = cik(A.kx[min(k, A1 - 1)], a);
            b = cik(A.kx[min(M - k, A1 - 1)], b);
        }
        if (k == 0) a.y = 0;  // c2r ignores the imaginary part of the DC term
        V* L = buf + t * LDP;
        const V w = wt[k];
        const V s = mkc<T>(a.x + b.x, a.y - b.y), d = mkc<T>(a.x - b.x, a.y + b.y);
        const V o = cmulc(d, w);
        L[k] = mkc<T>(s.x - o.y, s.y + o.x);
        if (k > 0 && 2 * k < M) L[M - k] = mkc<T>(s.x + o.y, o.x - s.y);
    }
    sync_lds();
    lds_fft_lines<T, M, NL, BS, +1, 1, false, xt_plan<M>()>(NL, [&](int line) { return buf + line * LDP; }, A.tw);
    constexpr int P = NL / 2;  // two levels per access
    for (int idx = threadIdx.x; idx < P * M; idx += BS) {
        const int u = idx % P;
        const int m = idx / P;
        const int z = z0 + 2 * u;
        if (z >= N3) continue;
        const V a = buf[2 * u * LDP + m], b = buf[(2 * u + 1) * LDP + m];
        T* o = out + (size_t(n2) * N1 + 2 * m) * N3 + z;
        *reinterpret_cast<V*>(o) = mkc<T>(a.x, b.x);
        *reinterpret_cast<V*>(o + N3) = mkc<T>(a.y, b.y);
    }
}

template <typename T, int N1>
__global__ __launch_bounds__(BS) void k_x_r2c(XTArgs<T> A) {
    using V = cx<T>;
    constexpr int M = N1 / 2, LDP = xt_ldp<M>(), NL = xt_levels<T, N1>();
    __shared__ V buf[NL * LDP];
    const int tile = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int n2 = tile / gridDim.x, z0 = (tile % gridDim.x) * NL;
    const int N3 = A.N3, A1 = A.A1;
    const T* __restrict__ in = A.nodal[blockIdx.z];
    V* __restrict__ out = A.spec[blockIdx.z];
    const V* __restrict__ wt = A.tw + 2 * M;
    constexpr int P = NL / 2;  // two levels per access
#pragma unroll 4
    for (int idx = threadIdx.x; idx < P * M; idx += BS) {
        const int u = idx % P;
        const int m = idx / P;
        const int z = z0 + 2 * u;
        V a = czero<V>(), b = czero<V>();
        if (z < N3) {
            const T* i = in + (size_t(n2) * N1 + 2 * m) * N3 + z;
            a = *reinterpret_cast<const V*>(i);
            b = *reinterpret_cast<const V*>(i + N3);
        }
        buf[2 * u * LDP + m] = mkc<T>(a.x, b.x);
        buf[(2 * u + 1) * LDP + m] = mkc<T>(a.y, b.y);
    }
    sync_lds();
    lds_fft_lines<T, M, NL, BS, -1, 1, false, xt_plan<M>()>(NL, [&](int line) { return buf + line * LDP; }, A.tw);
    const T h = T(0.5) * A.scale;
    for (int idx = threadIdx.x; idx < NL * A1; idx += BS) {
        const int t = idx / A1;
        const int k = idx - t * A1;
        const int z = z0 + t;
        if (z >= N3) continue;
        // X_k = (Z_k + conj Z_{M-k})/2 - i w^k (Z_k - conj Z_{M-k})/2
        const V Z = buf[t * LDP + k], W = buf[t * LDP + (k ? M - k : 0)];
        const V s = mkc<T>(Z.x + W.x, Z.y - W.y), d = mkc<T>(Z.x - W.x, Z.y + W.y);
        const V o = cmul(d, wt[k]);
        out[sidx(n2, z, k, N3, A1)] = mkc<T>(h * (s.x + o.y), h * (s.y - o.x));
    }
}

// spec = scale*(F(a) + ikx F(b)): a transform of b whose modes wait in registers
// for the transform of a, so that a sum of two nodal fields leaves as one
// spectrum
template <typename T, int N1>
__global__ __launch_bounds__(BS) void k_x_sum(XSumArgs<T> A) {
    using V = cx<T>;
    constexpr int M = N1 / 2, LDP = xt_ldp<M>(), NL = xt_levels<T, N1>();
    constexpr int PER = (NL * (N1 / 3) + BS - 1) / BS;  // modes per thread
    __shared__ V buf[NL * LDP];
    const int tile = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int n2 = tile / gridDim.x, z0 = (tile % gridDim.x) * NL;
    const int N3 = A.N3, A1 = A.A1;
    const V* __restrict__ wt = A.tw + 2 * M;
    V sum[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) sum[i] = czero<V>();
    const T h = T(0.5) * A.scale;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const T* in = pass == 0 ? A.b[blockIdx.z] : A.a[blockIdx.z];
        if (in == nullptr) continue;  // block-uniform
        constexpr int P = NL / 2;
#pragma unroll 4
        for (int idx = threadIdx.x; idx < P * M; idx += BS) {
            const int u = idx % P;
            const int m = idx / P;
            const int z = z0 + 2 * u;
            V a = czero<V>(), b = czero<V>();
            if (z < N3) {
                const T* i = in + (size_t(n2) * N1 + 2 * m) * N3 + z;
                a = *reinterpret_cast<const V*>(i);
                b = *reinterpret_cast<const V*>(i + N3);
            }
            buf[2 * u * LDP + m] = mkc<T>(a.x, b.x);
            buf[(2 * u + 1) * LDP + m] = mkc<T>(a.y, b.y);
        }
        sync_lds();
        lds_fft_lines<T, M, NL, BS, -1, 1, false, xt_plan<M>()>(NL, [&](int line) { return buf + line * LDP; }, A.tw);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = int(threadIdx.x) + i * BS;
            const int t = idx / A1;
            const int k = idx - t * A1;
            if (t >= NL) continue;
            const V Z = buf[t * LDP + k], W = buf[t * LDP + (k ? M - k : 0)];
            const V s = mkc<T>(Z.x + W.x, Z.y - W.y), d = mkc<T>(Z.x - W.x, Z.y + W.y);
            const V o = cmul(d, wt[k]);
            const V x = mkc<T>(h * (s.x + o.y), h * (s.y - o.x));
            if (pass == 0) {
                sum[i] = cik(A.kx[k], x);
            } else if (z0 + t < N3) {
                A.spec[blockIdx.z][sidx(n2, z0 + t, k, N3, A1)] = cadd(sum[i], x);
            }
        }
        sync_lds();
    }
}

template <typename T>
hipError_t launch_x_sum(const XSumArgs<T>& a, int N1, int N2, hipStream_t s) {
    if (a.nf < 1 || a.nf > XS_MAX || a.N3 % 2 != 0 || a.A1 > N1 / 3) return hipErrorInvalidValue;
    switch (N1) {
#define SF_CASE(n)                                                                                                 \
    case n:                                                                                                        \
        hipLaunchKernelGGL((k_x_sum<T, n>), dim3((a.N3 + xt_levels<T, n>() - 1) / xt_levels<T, n>(), N2, a.nf),    \
                           dim3(BS), 0, s, a);                                                                     \
        return hipGetLastError();
        SF_SIZES(SF_CASE)
#undef SF_CASE
        default:
            return hipErrorInvalidValue;
    }
}

template <typename T, int N1>
static hipError_t launch_xt_n(const XTArgs<T>& a, int N2, bool c2r, hipStream_t s) {
    constexpr int NL = xt_levels<T, N1>();
    const dim3 grid((a.N3 + NL - 1) / NL, N2, a.nf);
    if (c2r)
        hipLaunchKernelGGL((k_x_c2r<T, N1>), grid, dim3(BS), 0, s, a);
    else
        hipLaunchKernelGGL((k_x_r2c<T, N1>), grid, dim3(BS), 0, s, a);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_xt(const XTArgs<T>& a, int N1, int N2, bool c2r, hipStream_t s) {
    if (a.nf < 1 || a.nf > XT_MAX || a.N3 % 2 != 0 || a.A1 > N1 / 3) return hipErrorInvalidValue;
    switch (N1) {
#define SF_CASE(n) \
    case n:        \
        return launch_xt_n<T, n>(a, N2, c2r, s);
        SF_SIZES(SF_CASE)
#undef SF_CASE
        default:
            return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_x_c2r(const XTArgs<T>& a, int N1, int N2, hipStream_t s) {
    return launch_xt<T>(a, N1, N2, true, s);
}
template <typename T>
hipError_t launch_x_r2c(const XTArgs<T>& a, int N1, int N2, hipStream_t s) {
    return launch_xt<T>(a, N1, N2, false, s);
}

// the table of A.tw: the N1/2-point FFT's (fft_twiddle_table, 2M entries), then
// w^k for k < M
void xt_twiddles(int n, double* re, double* im) {
    const int M = n / 2;
    switch (n) {
#define SF_CASE(N)                            \
    case N:                                   \
        fft_twiddle_table<N / 2, xt_plan<N / 2>()>(re, im); \
        break;
        SF_SIZES(SF_CASE)
#undef SF_CASE
        default:
            return;
    }
    for (int k = 0; k < M; ++k) {
        re[2 * M + k] = std::cos(2 * cpi * k / n);
        im[2 * M + k] = -std::sin(2 * cpi * k / n);
    }
}

#define SF_TRANSFORM_INST(T)                                                     \
    template hipError_t launch_x_c2r<T>(const XTArgs<T>&, int, int, hipStream_t); \
    template hipError_t launch_x_r2c<T>(const XTArgs<T>&, int, int, hipStream_t); \
    template hipError_t launch_x_sum<T>(const XSumArgs<T>&, int, int, hipStream_t);

SF_TRANSFORM_INST(float)
SF_TRANSFORM_INST(double)

}  // namespace sf
