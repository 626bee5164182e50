// sf_kernels.h -- kernel argument blocks and host launchers.
#pragma once
#include "sf_common.h"

namespace sf {


// Fused per-mode stage kernel (one wavefront per Fourier mode).
template <typename T>
struct ModalArgs {
    int N3, N3p, A1, A2, threeD;
    // the coefficient table by level, [ZC_COUNT][N3p], and in the order of the
    // columns' lanes: row c of level lane*M + t at (c*M + t)*64 + lane, M = rows per
    // lane (zero beyond N3)
    const T *zc, *zl;
    const T *kx, *ky, *kx2, *ky2;
    cx<T> *u1, *u2, *u3, *b, *p;
    const cx<T> *ro1, *ro2, *ro3, *roB;  // explicit terms of the previous stage (null: not read)
    cx<T> *rn1, *rn2, *rn3, *rnB;        // explicit terms of this stage (null: not stored)
    const cx<T> *n1, *n2, *n3, *nB;      // nonlinear terms from the transform path
    T hz, mh, hb, cv, cb, Ri, pmult;
    int mode;         // 0: full stage, 1: projection only (RemoveDivergence)
    int skip_linear;  // 1: n1..nB are the complete explicit terms (BuildRHSAdjoint)
    T* ubar;          // non-null: EvolveBackground, U_ (the ZC_UBAR row of zc) diffuses in place
};

// Position of element (row, z, j1) of every spectral array: row is the active
// y-mode ja of a modal field ([ja][z][j1]) or the spanwise point n2 of an
// x-spectral intermediate ([n2][z][j1]).  j1 is fastest, so the x transforms
// read and write whole contiguous rows of A1 values, the y transforms read and
// write runs of a j1 tile, and the modal kernels stage a tile of consecutive
// j1 modes through LDS.
__host__ __device__ inline size_t sidx(int row, int z, int j1, int N3, int A1) {
    return (size_t(row) * size_t(N3) + size_t(z)) * size_t(A1) + size_t(j1);
}

// Base state of the linearised products at one x point (U_ not included).
template <typename T>
struct alignas(16) XBase {
    T u1, u2, u3, b;
};
template <typename T>
struct XBaseArgs {
    int N3, A1;
    const cx<T>* in[4];  // x spectra of u1, u2, u3, b
    XBase<T>* out;       // [n2][z][x point]
    const cx<T>* tw;
};

// Fused inverse-x / products / forward-x kernel.
template <typename T>
struct XArgs {
    int N1, N3, N3p, A1, zch;            // zch: z levels per block
    int N2;                              // 3D: y points (rows of the outputs)
    int tiled;                           // 3D: outputs in tiles of 16 modes (ytile_idx)
    const cx<T>* in[4];                  // u1, u2, u3, b spectra
    cx<T>* out[8];                       // 3D: A1,A2,A3,AB,B1,B2,B3,BB ; 2D: Nl1,-,Nl3,NlB
    const T* zc;
    const T* kx;
    const cx<T>* tw;
    T scale;
    int linear;                          // 1: linearised products (BuildRHSLinear)
    const XBase<T>* base;                // linear: the base state (launch_xbase)
};

// y-direction transforms (3D): per (z, tile of consecutive j1).
template <typename T>
struct YArgs {
    int N3, A1, A2, nf;
    const cx<T>* in[8];
    cx<T>* out[8];
    const T* ky;      // A2 active wavenumbers (forward: i*ky*B term)
    const cx<T>* tw;
    T scale;
    int paired;       // forward: out[r] = scale*(F(in[2r]) + i ky F(in[2r+1]))
    int tiled;        // paired forward: inputs in tiles of 16 modes (ytile_idx)
    unsigned iky;     // inverse: bit f set: field f is the y derivative of in[f]
};

// Offset of (n2, z, j1) in an x-spectral field stored in tiles of 16 modes,
// [z][j1/16][n2][j1%16] (A1 a multiple of 16): what the 3D x-pass writes and
// the paired forward y transform reads when the grid allows it
// (yfwd_tiles), so that a y-transform block's 16-mode tile is one
// contiguous run of N2*16 values.
__host__ __device__ inline size_t ytile_idx(int n2, int z, int j1, int N2, int A1) {
    return ((size_t(z) * size_t(A1 >> 4) + size_t(j1 >> 4)) * size_t(N2) + size_t(n2)) * 16 + size_t(j1 & 15);
}

// x transforms of nf fields between nodal and x-spectral layouts.
constexpr int XT_MAX = 12;
template <typename T>
struct XTArgs {
    int N3, A1, nf;
    cx<T>* spec[XT_MAX];
    T* nodal[XT_MAX];
    const cx<T>* tw;  // xt_twiddles
    T scale;
    unsigned ikx;  // c2r: bit f set: field f is the x derivative of its spectrum
    const T* kx;
};
// forward x transforms of sums: spec[f] = scale*(F(a[f]) + ikx F(b[f])) (b null: F(a) alone)
constexpr int XS_MAX = 8;
template <typename T>
struct XSumArgs {
    int N3, A1, nf;
    const T* a[XS_MAX];
    const T* b[XS_MAX];
    cx<T>* spec[XS_MAX];
    const cx<T>* tw;
    const T* kx;
    T scale;
};

template <typename T>
hipError_t launch_modal(const ModalArgs<T>& a, hipStream_t s);
// the same for grids of few modes (sf_modal_cols.hip): one block per mode
template <typename T>
hipError_t launch_modal_cols(const ModalArgs<T>& a, hipStream_t s);
// whether it is the faster one, for a stage (step) or the projection alone
bool modal_cols_fit(int A1, int A2, int N3, int value_bytes, bool step);
template <typename T>
hipError_t launch_xpass(const XArgs<T>& a, int N1, int N2, bool threeD, hipStream_t s);
template <typename T>
hipError_t launch_xbase(const XBaseArgs<T>& a, int N1, int N2, bool threeD, hipStream_t s);
// many independent 2D runs per launch: args and items live in device memory,
// items[i] = (run, work item of the run: x-pass z-block, modal tile of modes);
// grid-stride loop over `grid` blocks.  (A table of the items, since a search in
// the runs' first items is a chain of dependent loads before a block can start.)  The
// _batch launches take runs of one N1 (x-pass) or one rows-per-lane M
// (modal); the _mixed launches take runs of any N1 / N3, the modal one with
// mb (4 or 8) modes per block for every run.
template <typename T>
hipError_t launch_modal_batch(const ModalArgs<T>* args, const int2* items, int total, int M, int grid,
                              hipStream_t s);
template <typename T>
hipError_t launch_xpass_batch(const XArgs<T>* args, const int2* items, int total, int N1, int grid,
                              hipStream_t s);
// (mmax: the largest rows per lane of the runs; nmax: the largest N1)
template <typename T>
hipError_t launch_modal_mixed(const ModalArgs<T>* args, const int2* items, int total, int mb, int mmax,
                              int grid, hipStream_t s);
// (r1f: first radix of the FFT plans, 0 for the defaults or 8; each run's tw
// must be the table of its N1 under that plan, fft_twiddles_plan)
template <typename T>
hipError_t launch_xpass_mixed(const XArgs<T>* args, const int2* items, int total, int nmax, int r1f,
                              int grid, hipStream_t s);
template <typename T>
hipError_t launch_yinv(const YArgs<T>& a, int N2, hipStream_t s);
template <typename T>
hipError_t launch_yfwd(const YArgs<T>& a, int N2, hipStream_t s);
template <typename T>
hipError_t launch_x_c2r(const XTArgs<T>& a, int N1, int N2, hipStream_t s);
template <typename T>
hipError_t launch_x_r2c(const XTArgs<T>& a, int N1, int N2, hipStream_t s);
template <typename T>
hipError_t launch_x_sum(const XSumArgs<T>& a, int N1, int N2, hipStream_t s);
// FP64 inner products (sf_fields.hip): up to DOT_MAX pairs per call, the
// results in pinned host memory
constexpr int DOT_MAX = 4;
constexpr int DOT_BLOCKS = 1024;  // blocks (partial sums) per pair
constexpr int DOT_HOST = 32;      // up to here the host adds the blocks' sums
// A double as two words that each carry the number of the call it belongs to,
// so that the host can tell when both halves have arrived.
struct DotWord {
    unsigned long long half[2];  // bits 32..63: a half of the double, 0..31: the call
};
struct DotResult {
    DotWord sum[DOT_MAX][DOT_HOST];
};
// sums the host finds for each pair: the blocks' own, or their total
int dot_sums(size_t n);
template <typename T>
struct DotArgs {
    const cx<T>* a[DOT_MAX];
    const cx<T>* b[DOT_MAX];
    const T* w[DOT_MAX];  // vertical weights of each pair
    unsigned n, A1, N3;   // n = A1*A2*N3 values per field
    double* partial;      // DOT_MAX * DOT_BLOCKS values
    DotResult* host;
    unsigned call;        // number of the call
};
template <typename T>
hipError_t launch_dot(const DotArgs<T>& a, int pairs, hipStream_t s);
// copies of up to COPY_MAX modal fields in one launch (sf_fields.hip)
constexpr int COPY_MAX = 5;
enum CopyEnds { COPY_PLAIN = 0, COPY_NEUMANN, COPY_DIRICHLET };  // end conditions put on the copy (EnforceBCs)
template <typename T>
struct CopyArgs {
    const cx<T>* src[COPY_MAX];  // null: the copy is zero
    cx<T>* dst[COPY_MAX];
    int ends[COPY_MAX];
    unsigned n, A1, N3;  // n = A1*A2*N3 values per field, even (N3 is)
};
template <typename T>
hipError_t launch_copy(const CopyArgs<T>& a, int fields, hipStream_t s);
template <typename T>
hipError_t launch_maxabs(const T* f, size_t n, int N3, const T* add, double* partial, double* out, int slot,
                         hipStream_t s);
template <typename T>
hipError_t launch_axpby(cx<T>* y, T a, const cx<T>* x, T b, size_t n, hipStream_t s);
template <typename T>
hipError_t launch_ends(cx<T>* f, int A1, int A2, int N3, int bc_op, hipStream_t s);
template <typename T>
hipError_t launch_dmul(cx<T>* out, const cx<T>* in, int A1, int A2, int N3, const T* kx, const T* ky, int axis,
                       const T* zc, int N3p, hipStream_t s);

// diffusion preconditioner of the Newton-Krylov solves (one wavefront per mode)
template <typename T>
struct DiffPrecArgs {
    int N3, N3p, A1, A2, dirichlet;
    const T* zc;
    const T *kx, *kx2, *ky2;  // kx, -kx^2, -ky^2 of the active modes
    const cx<T>* in;
    cx<T>* out;
    T tnu, delta, k2max;
    T tadv;  // T of the advection term -i kx U(z) (0: diffusion only)
};
template <typename T>
hipError_t launch_diffprec(const DiffPrecArgs<T>& p, hipStream_t s);
// tadv != 0 (sf_precond.hip), for columns of up to advprec_rows levels
template <typename T>
constexpr int advprec_rows() {
    return sizeof(T) == 4 ? 512 : 256;
}
template <typename T>
hipError_t launch_advprec(const DiffPrecArgs<T>& p, hipStream_t s);

// adjoint step (sf_adjoint.hip)
template <typename T>
struct AdjArgs {
    int N3, N3p, A1;
    size_t n;            // nodal points N1*N2*N3
    const T* U[4];       // adjoint nodal u1, u2, u3, b
    const T* Tt[4];      // direct totals, nodal
    const T* DX[4];      // nodal ddx of the totals
    const T* DY[4];      // nodal ddy of the totals (3D)
    const cx<T>* u3t;    // modal totals, for the horizontal averages
    const cx<T>* bt;
    const T* zc;
    T Ri;
    T* Q[12];            // nodal explicit terms
};
// direct state at a stage: out[i] = (1-f) above[i] + f below[i], plus U_ on u1
template <typename T>
struct AdjLerp {
    int N3, A1, A2;
    unsigned n;  // A1*A2*N3
    T f;
    const T* ubar;
    const cx<T>* above[4];
    const cx<T>* below[4];
    cx<T>* out[4];  // null: absent
};
template <typename T>
hipError_t launch_adj_lerp(const AdjLerp<T>& a, hipStream_t s);
template <typename T>
hipError_t launch_add_profile(T* f, const T* prof, size_t n, int N3, hipStream_t s);
template <typename T>
hipError_t launch_adj_products(const AdjArgs<T>& a, bool three, hipStream_t s);
template <typename T>
hipError_t launch_mix_product(T* out, const T* Bt, const T* Wt, const cx<T>* bt, size_t n, int N3, int A1,
                              hipStream_t s);
template <typename T>
hipError_t launch_mean_profile(const cx<T>* f, double* out, int N3, int A1, hipStream_t s);
template <typename T>
hipError_t launch_phase_shift(cx<T>* f, size_t n, int A1, double shift, hipStream_t s);
template <typename T>
hipError_t launch_add_mean(cx<T>* f, int N3, int A1, T value, hipStream_t s);

bool tz_supported(int n);
// z levels per x-pass block for this grid (the block height that minimises
// rounds of resident blocks x (levels + 2))
int xpass_levels(int N1, int N2, int N3, bool threeD, bool linear, int precision);
// twiddle table of an n-point LDS FFT: 2n entries (the layout its second pass
// reads, then the same values in the order of the second pass on lane pairs)
void fft_twiddles(int n, double* re, double* im);
// the same for the plan with first radix r1f (8 or 16 where n allows it,
// else the default), and that plan's first radix
void fft_twiddles_plan(int n, int r1f, double* re, double* im);
// the paired forward y transform of this grid runs on tiles of 16 modes read
// as contiguous runs (A1 a multiple of 16 and k_yfwd_seq's LDS tile fits)
bool yfwd_tiles(int N2, int A1, int precision);
int fft_first_radix(int n, int r1f);
// the table of the whole-field x transforms: 3n/2 entries
void xt_twiddles(int n, double* re, double* im);
int max_rows_per_lane();
// blocks (and so partial maxima) of the two-pass max-abs reduction
int max_reduction_blocks();
// modes per block of the modal kernels for M rows per lane
int modal_modes_per_block(int M, int precision);

}  // namespace sf
