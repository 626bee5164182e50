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
// A 2D field is 0.2-0.7 MB, so latency and launches bound this, not HBM: the
// separate finishing kernel, the copy of the result to the host and the wait
// on the stream cost more than the sums.  Every block stores its partial sum
// and draws a ticket; the block with the last ticket adds the partials in
// block order (the same bits on every call) and writes the results and then
// the call's sequence number to pinned host memory, which the host reads.
// Partials and ticket go through agent-scope accesses, since the blocks run
// on XCDs with separate L2s.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(FB) void k_dot(DotArgs<T> A) {
    __shared__ double red[FB / 64];
    __shared__ bool last;
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
    unsigned e = blockIdx.x * FB + threadIdx.x;
    for (; e < n && n - e > 3 * stride; e += 4 * stride) {  // four elements in flight
        cx<T> x[4], v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = a[e + i * stride];
            v[i] = b[e + i * stride];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc += term(e + i * stride, x[i], v[i]);
    }
    for (; e < n; e += stride) acc += term(e, a[e], b[e]);
    acc = wave_sum(acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
#pragma unroll
        for (int i = 0; i < FB / 64; ++i) s += red[i];
        __hip_atomic_store(A.partial + y * gridDim.x + blockIdx.x, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned t = __hip_atomic_fetch_add(A.ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        last = t + 1 == gridDim.x * gridDim.y;
    }
    __syncthreads();
    if (!last) return;  // block-uniform
    // one wave per pair
    if (wave < int(gridDim.y)) {
        double s = 0;
        for (unsigned i = lane; i < gridDim.x; i += 64)
            s += __hip_atomic_load(A.partial + wave * gridDim.x + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s = wave_sum(s);
        if (lane == 0) __hip_atomic_store(&A.host->val[wave], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_store(A.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
        __hip_atomic_store(&A.host->seq, A.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Blocks per pair: four elements a thread, so that the 2D fields (some
// thousand modes and levels) take a few dozen blocks and the last one has few
// partials to add, up to DOT_BLOCKS where HBM bandwidth sets the time.
template <typename T>
hipError_t launch_dot(const DotArgs<T>& a, int pairs, hipStream_t s) {
    static_assert(DOT_MAX <= FB / 64, "the last block adds one pair per wave");
    if (pairs < 1 || pairs > DOT_MAX) return hipErrorInvalidValue;
    unsigned blocks = unsigned((a.n + 4 * FB - 1) / (4 * FB));
    if (blocks > unsigned(DOT_BLOCKS)) blocks = DOT_BLOCKS;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL((k_dot<T>), dim3(blocks, pairs), dim3(FB), 0, s, a);
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
