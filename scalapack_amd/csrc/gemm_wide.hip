// gemm_wide.hip -- C[m x n] -= A[m x k] * B[k x n] in FP64 with larger tiles than
// gemm_tile.hip's, for the trailing updates that outlast the panel beside them and
// for large products alone on the GPU.
//
// Bound by the matrix cores.  A 512-thread workgroup, one a CU, takes a 128 x 256 tile,
// two waves a SIMD, so per flop it moves a third of what 64 x 64 tiles move through
// the L2 and LDS, and reaches a higher rate where it has many tiles and runs for long:
// m = n = 16384, k = 1024: 62.2 TF/s, 59.8 with 64 x 64 tiles; k = 512 57.7, 57.3; inside the
// factorization at N = 32768, NB = 512, first update: 52.8 TF/s beside the panel, 47
// (three 64 x 64 workgroups a CU, which leave the panel room) and 52 (four).  But it
// keeps a panel's kernels waiting for a CU to finish a tile, so an update that does not
// outlast its panel goes to gemm_tile_sub.
#include "sla_common.h"
#include "sla_kernels.h"

#include <cstdint>

namespace sla {

namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));

// Tile of a linear workgroup id: the ids an XCD receives (congruent mod 8) take a
// contiguous range of tiles, down the rows of bands of 8 tile columns.
__device__ __forceinline__ void tile_coords(int id, int tiles_m, int tiles_n, int &tm, int &tn)
{
    const int total = tiles_m * tiles_n, per = total / 8, rem = total % 8, x = id % 8;
    const int lid = x * per + min(x, rem) + id / 8;
    const int band = 8, full = tiles_n / band * band;
    if (lid < full * tiles_m) {
        const int r = lid % (band * tiles_m);
        tm = r % tiles_m;
        tn = lid / (band * tiles_m) * band + r / tiles_m;
    } else {
        const int r = lid - full * tiles_m;
        tm = r % tiles_m;
        tn = full + r / tiles_m;
    }
}

// A (128 x 16) and B (16 x 256) of each 16-deep K step are staged once in
// double-buffered LDS and shared by the eight waves, each with a 64 x 64 part of the
// tile as 4 x 4 accumulators; the next step's global loads are in flight during this
// step's MFMAs.  The A rows are stored permuted (LDS position 16 i + l of a wave's 64
// rows holds its row 4 l + i), so MFMA block i's operand row l is C row 4 l + i and a
// lane's four outputs of element r are four consecutive rows: one 32-byte access of C
// each.  Requires m a multiple of 128, n of 256, k of 16, and 32-byte aligned columns.
// The grid may be smaller than the number of tiles, then a multiple of 8 (as in
// gemm_tile.hip).
constexpr int XM = 128, XN = 256, XK = 16, XT = 512;

template <int TRAILING>
__global__ __launch_bounds__(XT, 1) void dgemm_nn_sub_wide_kernel(
    int m, int n, int k, const double *__restrict__ A, int lda, const double *__restrict__ B,
    int ldb, double *__restrict__ C, int ldc, unsigned long long *stamp)
{
    __shared__ __align__(16) double As[2][XK][XM];
    __shared__ __align__(16) double Bs[2][XK][XN];
    launch_stamp_begin(stamp);
    const int tiles_m = m / XM, tiles_n = n / XN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
    // global -> register: A rows a_r .. a_r + 3 at k = a_k; B column b_c,
    // k = b_k .. b_k + 7
    const int a_r = 4 * (tid & 31), a_k = tid >> 5;
    const int a_pos = (a_r / 64) * 64 + (a_r % 64) / 4;  // + 16 e for row a_r + e
    const int b_c = tid & 255, b_k = (tid >> 8) * 8;
    const int nk = k / XK;
    for (int tile = blockIdx.x; tile < tiles_m * tiles_n; tile += gridDim.x) {
        int tmi, tni;
        tile_coords(tile, tiles_m, tiles_n, tmi, tni);
        const int bm = tmi * XM, bn = tni * XN;
        const double *Ap = A + bm + a_r + (size_t)a_k * lda;
        const double *Bp = B + (size_t)(bn + b_c) * ldb + b_k;
        d4_t ra, rb[2];
        auto gload = [&](int kt) {
            const size_t k0 = (size_t)kt * XK;
            ra = *(const d4_t *)(Ap + k0 * lda);
            rb[0] = *(const d4_t *)(Bp + k0);
            rb[1] = *(const d4_t *)(Bp + k0 + 4);
        };
        auto lstore = [&](int buf) {
#pragma unroll
            for (int e = 0; e < 4; e++) As[buf][a_k][a_pos + 16 * e] = ra[e];
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) Bs[buf][b_k + 4 * q + e][b_c] = rb[q][e];
        };
        d4_t acc[4][4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
        gload(0);
        lstore(0);
        __syncthreads();
        for (int kt = 0; kt < nk; kt++) {
            const int buf = kt & 1;
            if (kt + 1 < nk) gload(kt + 1);
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                double a[4], b[4];
#pragma unroll
                for (int i = 0; i < 4; i++) a[i] = As[buf][4 * s4 + lk][wm + 16 * i + lr];
#pragma unroll
                for (int j = 0; j < 4; j++) b[j] = Bs[buf][4 * s4 + lk][wn + 16 * j + lr];
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
            }
            if (kt + 1 < nk) lstore(buf ^ 1);
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            double *Cc = C + (size_t)(bn + wn + 16 * j + lr) * ldc + bm + wm;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                d4_t *cp = (d4_t *)(Cc + 4 * (lk + 4 * r));
                d4_t c = *cp;
                c[0] -= acc[0][j][r];
                c[1] -= acc[1][j][r];
                c[2] -= acc[2][j][r];
                c[3] -= acc[3][j][r];
                *cp = c;
            }
        }
    }
    launch_stamp_end(stamp);
}

// No LDS and no workgroup barrier: a 128 x 128 tile per 256-thread workgroup, one a
// CU, each wave a 64 x 64 part whose operands it loads itself, three 16-deep K steps in
// flight.  Two index permutations make every lane's operands 32 contiguous bytes:
//   rows : MFMA block i, operand row lr  <->  C row wm + 4 lr + i
//   K    : operand k-lane lk, step s     <->  k = k0 + 4 lk + s
// A and B use the same K permutation; D element r of lane l (block row l / 16 + 4 r) is C
// row wm + 4 (l / 16 + 4 r) + i, four consecutive rows for i = 0 .. 3.  Requires m, n
// multiples of 128, k of 16, and 32-byte aligned columns.
constexpr int DEPTH = 3;

__global__ __launch_bounds__(256, 1) void dgemm_nn_sub_direct_kernel(
    int m, int n, int k, const double *__restrict__ A, int lda,
    const double *__restrict__ B, int ldb, double *__restrict__ C, int ldc)
{
    int tmi, tni;
    tile_coords(blockIdx.x, m / 128, n / 128, tmi, tni);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = tmi * 128 + (wave & 1) * 64, wn = tni * 128 + (wave >> 1) * 64;
    const int lr = lane & 15, lk = lane >> 4;
    const double *Ap = A + (wm + 4 * lr) + (size_t)(4 * lk) * lda;
    const double *Bp = B + (size_t)(wn + lr) * ldb + 4 * lk;
    const size_t bstep = (size_t)16 * ldb;

    d4_t a[DEPTH][4], b[DEPTH][4];
    auto load = [&](int t, int q) {
        const size_t k0 = (size_t)16 * t;
#pragma unroll
        for (int s = 0; s < 4; s++) a[q][s] = *(const d4_t *)(Ap + (k0 + s) * lda);
#pragma unroll
        for (int j = 0; j < 4; j++) b[q][j] = *(const d4_t *)(Bp + j * bstep + k0);
    };
    d4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};

    const int nk = k / 16;
#pragma unroll
    for (int q = 0; q < DEPTH - 1; q++)
        if (q < nk) load(q, q);
    for (int t = 0; t < nk; t += DEPTH) {
#pragma unroll
        for (int q = 0; q < DEPTH; q++) {
            if (t + q < nk) {
                const int nt = t + q + DEPTH - 1;
                if (nt < nk) load(nt, (q + DEPTH - 1) % DEPTH);
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q][s][i], b[q][j][s],
                                                                            acc[i][j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        double *Cc = C + (size_t)(wn + 16 * j + lr) * ldc;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            d4_t *cp = (d4_t *)(Cc + wm + 4 * (lk + 4 * r));
            d4_t c = *cp;
            c[0] -= acc[0][j][r];
            c[1] -= acc[1][j][r];
            c[2] -= acc[2][j][r];
            c[3] -= acc[3][j][r];
            *cp = c;
        }
    }
}

// What both kernels require of the operands.
bool aligned32(int k, const double *A, int lda, const double *B, int ldb, const double *C, int ldc)
{
    auto ok = [](const double *p, int ld) {
        return (reinterpret_cast<uintptr_t>(p) & 31) == 0 && ld % 4 == 0;
    };
    return k > 0 && k % 16 == 0 && ok(A, lda) && ok(B, ldb) && ok(C, ldc);
}

}  // namespace

bool gemm_wide_sub(int m, int n, int k, const double *A, int lda, const double *B, int ldb,
                   double *C, int ldc, hipStream_t s, int max_wgs, unsigned long long *stamp)
{
    const int mw = m / XM * XM, nw = n / XN * XN;
    if (mw <= 0 || nw <= 0 || !aligned32(k, A, lda, B, ldb, C, ldc)) return false;
    const int tiles = (mw / XM) * (nw / XN);
    const int grid = max_wgs >= 8 && tiles > max_wgs ? max_wgs / 8 * 8 : tiles;
    hipLaunchKernelGGL(dgemm_nn_sub_wide_kernel<1>, dim3(grid), dim3(XT), 0, s, mw, nw, k, A, lda, B,
                       ldb, C, ldc, stamp);
    SLA_LAUNCH_CHECK();
    // the rows below the tiles (all columns) and the columns right of them
    gemm_tile_sub<double>(false, m - mw, n, k, A + mw, lda, B, ldb, C + mw, ldc, s, true,
                          GEMM_TILE_WGS_PER_CU * max_wgs, false, stamp);
    gemm_tile_sub<double>(false, mw, n - nw, k, A, lda, B + (size_t)nw * ldb, ldb,
                          C + (size_t)nw * ldc, ldc, s, true, GEMM_TILE_WGS_PER_CU * max_wgs, false,
                          stamp);
    return true;
}

void dgemm_alone_sub(int m, int n, int k, const double *A, int lda, const double *B, int ldb,
                     double *C, int ldc, hipStream_t s, int cus)
{
    // The larger tiles are worth their while for long sums and where a tile a CU
    // leaves hardly any CU idle in the last round.  TF/s with tiles of 64 x 64, 128 x
    // 128, 128 x 256: m = n = 2048, k = 512 41, 44, 27; k = 4096 53, 63, 33; 3072, k =
    // 4096 (2.25 rounds) 55, 50, 37; 4096, k = 512 54, 56, 56; k = 4096 60, 65, 65; 6144, k =
    // 512 55, 52, 50; k = 2048 59, 63, 58; 12288, k = 512 57, 54, 57; k = 1024 59, 60, 62.
    auto full = [&](int t) { return t >= 0.95 * cus * ceil_div(t, cus); };
    const int md = m / 128 * 128, nd = n / 128 * 128;
    const int wide = (m / XM) * (n / XN), direct = (md / 128) * (nd / 128);
    if (k >= 1024 && wide > 0 && full(wide) && gemm_wide_sub(m, n, k, A, lda, B, ldb, C, ldc, s, 0, nullptr))
        return;
    if (direct > 0 && full(direct) && (k >= 1024 || (k >= 512 && direct <= 4 * cus)) &&
        aligned32(k, A, lda, B, ldb, C, ldc)) {
        hipLaunchKernelGGL(dgemm_nn_sub_direct_kernel, dim3(direct), dim3(256), 0, s, md, nd, k, A,
                           lda, B, ldb, C, ldc);
        SLA_LAUNCH_CHECK();
        gemm_tile_sub<double>(false, m - md, n, k, A + md, lda, B, ldb, C + md, ldc, s);
        gemm_tile_sub<double>(false, md, n - nd, k, A, lda, B + (size_t)nd * ldb, ldb,
                              C + (size_t)nd * ldc, ldc, s);
        return;
    }
    gemm_tile_sub<double>(false, m, n, k, A, lda, B, ldb, C, ldc, s);
}

}  // namespace sla
