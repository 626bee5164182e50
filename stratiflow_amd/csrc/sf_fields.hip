// sf_fields.hip -- whole-field kernels behind the StateVector algebra: FP64
// inner products and copies between states.
#include "sf_kernels.h"

namespace sf {

namespace {
constexpr int FB = 256;  // threads per block

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
    return v;
}
}  // namespace

// ---------------------------------------------------------------------------
// FP64 inner products, InnerProd (Integration.h:117-146):
//   sum_z w_z sum_modes c_m Re(a conj b),  c = 1 for mode (0,0), 2 otherwise,
// of up to DOT_MAX field pairs (blockIdx.y) in one launch.
//
// A 2D field is 0.2-0.7 MB, so latency and launches bound this, not HBM: a
// separate finishing kernel, the copy of the result to the host and the wait
// on the stream cost more than the sums.  Results go straight to pinned host
// memory, which the host watches.  Up to DOT_HOST blocks each write their own sum
// and the host adds them; the partials of more blocks are added by a second launch.
// (A ticket by which the last block adds them is one atomic per block on one
// address: the four pairs of an energy of 384x192x384 FP32 took 168 us with it,
// 49 without, one pair 47 and 23; 512x1x512 FP32 takes 13 and 11.)
// Either way the sums are added in a fixed order: the same bits on every call.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void dot_send(DotWord* to, double v, unsigned call) {
    const unsigned long long b = __double_as_longlong(v);
    __hip_atomic_store(&to->half[0], (b << 32) | call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&to->half[1], (b >> 32 << 32) | call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename T>
__global__ __launch_bounds__(FB) void k_dot(DotArgs<T> A) {
    __shared__ double red[FB / 64];
    const int y = blockIdx.y;
    const cx<T>* __restrict__ a = A.a[y];
    const cx<T>* __restrict__ b = A.b[y];
    const T* __restrict__ w = A.w[y];
    const unsigned n = A.n, A1 = A.A1, N3 = A.N3;
    const unsigned stride = gridDim.x * FB;
    double acc = 0;
    auto term = [&](unsigned e, cx<T> x, cx<T> v) {
        const unsigned rowz = e / A1;  // [ja][z][j1]
        const unsigned z = rowz % N3;
        const bool m00 = rowz < N3 && e == rowz * A1;  // ja == 0 and j1 == 0
        const double re = double(x.x) * double(v.x) + double(x.y) * double(v.y);
        return (m00 ? 1.0 : 2.0) * double(w[z]) * re;
    };
    // four elements in flight; past the end the first one with a zero factor, so
    // that the last round is no chain of single loads
    for (unsigned e = blockIdx.x * FB + threadIdx.x; e < n; e += 4 * stride) {
        cx<T> x[4], v[4];
        unsigned at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            at[i] = n - e > i * stride ? e + i * stride : e;
            x[i] = a[at[i]];
            v[i] = b[at[i]];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double t = term(at[i], x[i], v[i]);
            acc += i == 0 || at[i] != e ? t : 0.0;
        }
    }
    acc = wave_sum(acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
#pragma unroll
        for (int i = 0; i < FB / 64; ++i) s += red[i];
        if (gridDim.x <= DOT_HOST) dot_send(&A.host->sum[y][blockIdx.x], s, A.call);
        else A.partial[y * gridDim.x + blockIdx.x] = s;
    }
}

// one wave per pair adds its partials
static __global__ __launch_bounds__(64) void k_dot_sum(const double* __restrict__ partial, int blocks, DotResult* host,
                                                       unsigned call) {
    const int y = blockIdx.x;
    double s = 0;
    for (int i = threadIdx.x; i < blocks; i += 64) s += partial[y * blocks + i];
    s = wave_sum(s);
    if (threadIdx.x == 0) dot_send(&host->sum[y][0], s, call);
}

// Blocks per pair: four elements a thread, up to DOT_BLOCKS where HBM bandwidth
// sets the time; fields of up to 16 elements a thread of DOT_HOST blocks take those.
static unsigned dot_blocks(size_t n) {
    const size_t four = (n + 4 * FB - 1) / (4 * FB);
    if (four <= DOT_HOST) return four < 1 ? 1 : unsigned(four);
    if (n <= size_t(DOT_HOST) * FB * 16) return DOT_HOST;
    return unsigned(four < size_t(DOT_BLOCKS) ? four : size_t(DOT_BLOCKS));
}
int dot_sums(size_t n) {
    const unsigned b = dot_blocks(n);
    return b <= DOT_HOST ? int(b) : 1;
}

template <typename T>
hipError_t launch_dot(const DotArgs<T>& a, int pairs, hipStream_t s) {
    if (pairs < 1 || pairs > DOT_MAX) return hipErrorInvalidValue;
    const unsigned blocks = dot_blocks(a.n);
    hipLaunchKernelGGL((k_dot<T>), dim3(blocks, pairs), dim3(FB), 0, s, a);
    if (blocks > DOT_HOST)
        hipLaunchKernelGGL(k_dot_sum, dim3(pairs), dim3(64), 0, s, a.partial, int(blocks), a.host, a.call);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// A state's fields copied in one launch (blockIdx.y = field): CopyToSolver,
// CopyFromSolver with the end conditions of EnforceBCs (StateVector.h:415-421,
// 511-543), the populated snapshot, SetBackground.  Moving a 2D field takes
// less time than launching its copy, so five copies and four end-condition
// passes cost nine launches' time; here one.  16 bytes per thread and load; the
// level of an element is only needed where end conditions are.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(FB) void k_copy(CopyArgs<T> A) {
    using V = cx<T>;
    constexpr int NV = 16 / int(sizeof(V));  // values per thread and round
    struct alignas(16) Pack {
        V v[NV];
    };
    const int f = blockIdx.y;
    const V* src = A.src[f];  // may be dst (no restrict)
    V* dst = A.dst[f];
    const int ends = A.ends[f];
    const unsigned packs = A.n / NV, A1 = A.A1, N3 = A.N3;
    for (unsigned i = blockIdx.x * FB + threadIdx.x; i < packs; i += gridDim.x * FB) {
        Pack p;
        if (src) {
            p = reinterpret_cast<const Pack*>(src)[i];
            if (ends != COPY_PLAIN) {
#pragma unroll
                for (int q = 0; q < NV; ++q) {
                    const unsigned e = i * NV + q;
                    const unsigned z = (e / A1) % N3;
                    if (ends == COPY_NEUMANN) {
                        if (z == 0) p.v[q] = src[e + A1];
                        if (z == N3 - 1) p.v[q] = src[e - A1];
                    } else if (z <= 2 || z >= N3 - 2) {
                        p.v[q] = czero<V>();
                    }
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) p.v[q] = czero<V>();
        }
        reinterpret_cast<Pack*>(dst)[i] = p;
    }
}

template <typename T>
hipError_t launch_copy(const CopyArgs<T>& a, int fields, hipStream_t s) {
    if (fields < 1 || fields > COPY_MAX || a.n % 2 != 0) return hipErrorInvalidValue;
    unsigned blocks = (a.n / (16 / unsigned(sizeof(cx<T>))) + FB - 1) / FB;
    if (blocks > 2048) blocks = 2048;  // eight per CU
    hipLaunchKernelGGL((k_copy<T>), dim3(blocks, fields), dim3(FB), 0, s, a);
    return hipGetLastError();
}

#define SF_FIELDS_INST(T)                                                      \
    template hipError_t launch_dot<T>(const DotArgs<T>&, int, hipStream_t);    \
    template hipError_t launch_copy<T>(const CopyArgs<T>&, int, hipStream_t);

SF_FIELDS_INST(float)
SF_FIELDS_INST(double)

}  // namespace sf
