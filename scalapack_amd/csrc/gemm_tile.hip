// gemm_tile.hip -- C[m x n] -= op(A)[m x k] * B[k x n] on the matrix cores, any
// m, n, k and leading dimensions, op(A) = A or A^T: the trailing (Schur
// complement) update of the FP64 factorization, A22 <- A22 - L21 * U12, and the
// products inside the recursive panel, the block triangular solves and (FP32
// too) the low-precision factorization's panel.
//
// The trailing update is the one local dgemm_ PDGEMM issues on a 1 x 1 grid
// (SRC/pdgetrf.f:288-290 -> PBLAS/SRC/pdgemm_.c:476 ->
//  PBLAS/SRC/PTOOLS/PB_CpgemmAB.c:333-352: dgemm_('N','N', M-J-JB+1,
//  N-J-JB+1, JB, -1, L21, LLD, U12, LLD, +1, A22, LLD)).
//
// A 256-thread workgroup owns a 64 x BN tile of C (BN = 64 or 32), K in steps
// of 16 through double-buffered LDS, the next step's global loads in registers
// during this step's 16 x 16 x 4 MFMAs.  The instruction is given op(A)'s rows
// as its second operand and B's columns as its first, so that it leaves C^T in
// the accumulators: the 16 lanes of a row group hold 16 rows of one column and
// access 16 consecutive elements of C with plain loads and stores, whatever the
// alignment.  Rows and columns beyond the matrix are loaded from its last row or
// column and not stored; the steps beyond k are zeros in both operands.  The
// products are summed before C is subtracted from.
//
// FP64: bound by the matrix cores (64 cycles an instruction and SIMD, 78.6 TF/s)
// when they are kept busy.  That takes several waves a SIMD -- one wave's waits
// for LDS, global loads, the barrier and the tile's first and last accesses are
// another's MFMAs -- so the tile is small enough for four workgroups a CU (at
// most 128 registers, 33 KB of LDS), which also spreads small products over the
// chip and leaves room for a panel.  Larger tiles pay where many of them run for
// long (gemm_wide.hip).  128 x 64 in 256 threads was slower (39 TF/s where this one
// has 57), and so was loading C at the end, not at the start (54 against 58 TF/s).
// Measured, with the kernels of 128 x 256 and 128 x 128 tiles, and thin ones for n, k
// <= 64, that it replaced, and now, us: m = n = 16128, k = 512: 4715, 4605 (57.8
// TF/s); k = 256: 2710, 2487; 8192, k = 512: 1210, 1211; 4096, k = 512: 292, 303; 3072,
// k = 512: 290, 181; 2900, k = 128: 141, 59; 2900, k = 128, odd leading
// dimension: 107, 59; 960, k = 64: 99, 8; m x 32 x 32, m = 16384: 8.2, 4.2.
#include "sla_common.h"
#include "sla_kernels.h"

#include <algorithm>
#include <cstdint>
#include <type_traits>

namespace sla {

namespace {

constexpr int GM = 64, GK = 16, GT = 256;
typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4_t mfma(double a, double b, d4_t c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma(float a, float b, f4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Tile of a linear workgroup id: the ids an XCD receives (congruent mod 8)
// take a contiguous range of tiles, column bands of 8 tiles wide, so that
// neighbours in time share operands in the XCD's L2.
__device__ __forceinline__ void tile_of(int id, int tm, int tn, int &im, int &in)
{
    const int total = tm * tn, per = total / 8, rem = total % 8, x = id % 8, k = id / 8;
    const int lid = x * per + min(x, rem) + k;  // k < per + (x < rem)
    const int band = 8, full = tn / band * band;
    if (lid < full * tm) {
        const int r = lid % (band * tm);
        im = r / band;
        in = lid / (band * tm) * band + r % band;
    } else {
        const int r = lid - full * tm, w = tn - full;
        im = r / w;
        in = full + r % w;
    }
}

// USE distinguishes the launches of the outer trailing update from the others in
// kernel traces, and those of the solves, whose sums are of at most FOLD steps
// (128 products) each and subtracted from C one after another: of 256 products in
// one sum, PDGETRS's backward error was up to 1.2 times what it had been with four
// sums side by side (n = 700).  The trailing update's grid may be smaller than the
// tile count (a persistent launch that leaves CUs free): workgroup b takes tiles b,
// b + grid, ...; grid is then a multiple of 8, so a tile index keeps its XCD.
// O: type of the byte offsets within a tile's operands.
enum Use { PLAIN = 0, TRAILING = 1, SOLVE = 2 };
constexpr int FOLD = 8;

template <typename T, typename O, bool TA, int BN, int USE>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(4))) void gemm_tile_kernel(
    int m, int n, int k, const T *__restrict__ A, int lda, const T *__restrict__ B, int ldb,
    T *__restrict__ C, int ldc, unsigned long long *stamp)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, d4_t, f4_t>::type;
    // waves: BN = 64: 2 x 2 of 32 x 32; BN = 32: 4 x 1 of 16 x 32
    constexpr int NA = BN == 64 ? 2 : 1, NB = 2;  // 16 x 16 blocks of a wave
    constexpr int LA = GM * GK / GT, LB = BN * GK / GT;  // loads of a thread and step
    __shared__ T As[2][GK][GM + 1];
    __shared__ T Bs[2][GK][BN + 1];
    if (USE == TRAILING) launch_stamp_begin(stamp);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
    const int wm = BN == 64 ? (wave & 1) * 32 : wave * 16, wn = BN == 64 ? (wave >> 1) * 32 : 0;
    // column of C of accumulator element r within a 16 x 16 block
    auto ccol = [&](int r) { return sizeof(T) == 8 ? lk + 4 * r : 4 * lk + r; };
    const int tm = (m + GM - 1) / GM, tn = (n + BN - 1) / BN;
    for (int tile = blockIdx.x; tile < tm * tn; tile += USE == TRAILING ? gridDim.x : tm * tn) {
    int im, in;
    tile_of(tile, tm, tn, im, in);
    const int bm = im * GM, bn = in * BN;

    // Loads: op(A) = A: 64 rows of one k a wave; A^T and B: 16 k of a row or
    // column in 16 lanes.  A uniform pointer walks along k and every thread
    // keeps byte offsets from it, so that a step's loads need no address
    // arithmetic.
    const int kq = tid & 15, cq = tid >> 4;
    const T *Ak = A + (TA ? (size_t)bm * lda : (size_t)bm), *Bk = B + (size_t)bn * ldb;
    O oa[TA ? LA : 1], ob[LB];
    if constexpr (TA) {
#pragma unroll
        for (int i = 0; i < LA; i++)
            oa[i] = (O)sizeof(T) * ((O)min(cq + 16 * i, m - 1 - bm) * (O)lda + kq);
    } else {
        oa[0] = (O)sizeof(T) * ((O)(wave * LA) * (O)lda + min(lane, m - 1 - bm));
    }
#pragma unroll
    for (int i = 0; i < LB; i++)
        ob[i] = (O)sizeof(T) * ((O)min(cq + 16 * i, n - 1 - bn) * (O)ldb + kq);
    auto at = [](const T *p, O o) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + o);
    };
    auto at_a = [&](int i) { return TA ? at(Ak, oa[TA ? i : 0]) : at(Ak + (size_t)i * lda, oa[0]); };
    T ra[LA], rb[LB];
    auto load = [&](int left) {  // the next step, `left` of k still to come
        if (left >= GK) {
#pragma unroll
            for (int i = 0; i < LA; i++) ra[i] = at_a(i);
#pragma unroll
            for (int i = 0; i < LB; i++) rb[i] = at(Bk, ob[i]);
        } else {
#pragma unroll
            for (int i = 0; i < LA; i++) {
                const bool in = (TA ? kq : wave * LA + i) < left;
                ra[i] = in ? at_a(i) : T(0);
            }
#pragma unroll
            for (int i = 0; i < LB; i++) rb[i] = kq < left ? at(Bk, ob[i]) : T(0);
        }
        Ak += TA ? (size_t)GK : (size_t)GK * lda;
        Bk += GK;
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            if constexpr (TA) As[buf][kq][cq + 16 * i] = ra[i];
            else As[buf][wave * LA + i][lane] = ra[i];
        }
#pragma unroll
        for (int i = 0; i < LB; i++) Bs[buf][kq][cq + 16 * i] = rb[i];
    };

    acc_t acc[NA][NB], c[NA][NB];
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = acc_t{0, 0, 0, 0};
    load(k);
    // C is wanted last but loaded first: for a small k its latency is most of
    // the tile's time
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = min(bm + wm + 16 * i + lr, m - 1);
                const int col = min(bn + wn + 16 * j + ccol(r), n - 1);
                c[i][j][r] = C[(size_t)row + (size_t)col * ldc];
            }
    store(0);
    __syncthreads();
    const int nk = (k + GK - 1) / GK;
    for (int t = 0; t < nk; t++) {
        const int buf = t & 1;
        if (t + 1 < nk) load(k - (t + 1) * GK);
#pragma unroll
        for (int s = 0; s < GK / 4; s++) {
            T a[NA], b[NB];
#pragma unroll
            for (int i = 0; i < NA; i++) a[i] = As[buf][4 * s + lk][wm + 16 * i + lr];
#pragma unroll
            for (int j = 0; j < NB; j++) b[j] = Bs[buf][4 * s + lk][wn + 16 * j + lr];
#pragma unroll
            for (int i = 0; i < NA; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
                    acc[i][j] = mfma(b[j], a[i], acc[i][j]);
        }
        if (USE == SOLVE && (t + 1) % FOLD == 0) {
#pragma unroll
            for (int i = 0; i < NA; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    c[i][j] -= acc[i][j];
                    acc[i][j] = acc_t{0, 0, 0, 0};
                }
        }
        if (t + 1 < nk) store(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = bm + wm + 16 * i + lr, col = bn + wn + 16 * j + ccol(r);
                if (row < m && col < n)
                    C[(size_t)row + (size_t)col * ldc] = c[i][j][r] - acc[i][j][r];
            }
    }  // tile loop
    if (USE == TRAILING) launch_stamp_end(stamp);
}

}  // namespace

template <typename T>
void gemm_tile_sub(bool ta, int m, int n, int k, const T *A, int lda, const T *B, int ldb, T *C,
                   int ldc, hipStream_t s, bool trailing, int max_wgs, bool beside,
                   unsigned long long *stamp, bool solve)
{
    if (m <= 0 || n <= 0 || k <= 0) return;
    if (solve ? trailing || sizeof(T) != 8 : ta)
        throw std::logic_error("gemm: only the solves' products, in FP64, are transposed");
    // n <= 32 would leave half of a 64-wide tile empty
    const int tiles = ceil_div(m, GM) * ceil_div(n, n <= 32 ? 32 : 64);
    // only the trailing update's kernel takes several tiles a workgroup
    const int grid = trailing && max_wgs >= 8 && tiles > max_wgs ? max_wgs / 8 * 8 : tiles;
    // Beside a panel: LDS beyond the kernel's own, so that three workgroups (41 KB
    // each) share a CU and a fourth does not fit.  37 KB of LDS and a quarter of
    // the registers stay free for the panel's kernels, which otherwise wait until
    // the update has no more workgroups to start: it has one ready whenever a slot
    // is free.  The update alone gets 9 % slower (m = n = 16128, k = 512: 4574,
    // 4985 us); PDGETRF at N = 16384, NB = 256 takes 118 ms instead of 138.
    const unsigned lds = beside ? 8000 : 0;
    // offsets of 64 columns and a step in 32 bits, but for extreme leading dimensions
    const bool small = (size_t)(64 + GK) * std::max(lda, ldb) * sizeof(T) < (size_t)UINT32_MAX;
#define SLA_TILE(TAV, BNV, USEV)                                                                \
    do {                                                                                        \
        if (small)                                                                              \
            hipLaunchKernelGGL((gemm_tile_kernel<T, uint32_t, TAV, BNV, USEV>), dim3(grid),     \
                               dim3(GT), lds, s, m, n, k, A, lda, B, ldb, C, ldc, stamp);       \
        else                                                                                    \
            hipLaunchKernelGGL((gemm_tile_kernel<T, uint64_t, TAV, BNV, USEV>), dim3(grid),     \
                               dim3(GT), lds, s, m, n, k, A, lda, B, ldb, C, ldc, stamp);       \
    } while (0)
    if (trailing) {
        if (n <= 32) SLA_TILE(false, 32, TRAILING);
        else SLA_TILE(false, 64, TRAILING);
    } else if (!solve) {
        if (n <= 32) SLA_TILE(false, 32, PLAIN);
        else SLA_TILE(false, 64, PLAIN);
    } else if constexpr (sizeof(T) == 8) {
        if (n <= 32) {
            if (ta) SLA_TILE(true, 32, SOLVE);
            else SLA_TILE(false, 32, SOLVE);
        } else {
            if (ta) SLA_TILE(true, 64, SOLVE);
            else SLA_TILE(false, 64, SOLVE);
        }
    }
#undef SLA_TILE
    SLA_LAUNCH_CHECK();
}
template void gemm_tile_sub<double>(bool, int, int, int, const double *, int, const double *, int,
                                    double *, int, hipStream_t, bool, int, bool,
                                    unsigned long long *, bool);
template void gemm_tile_sub<float>(bool, int, int, int, const float *, int, const float *, int,
                                   float *, int, hipStream_t, bool, int, bool,
                                   unsigned long long *, bool);

}  // namespace sla
