// trsm.hip -- triangular solves of the LU path.
//
// trsm_llnu: the block row of U in PDGETRF, U12 <- L11^{-1} A12
//   (SRC/pdgetrf.f:280-281, PDTRSM('L','L','N','U'); on a 1 x 1 grid
//   PBLAS/SRC/PTOOLS/PB_CptrsmAB.c:359-412 splits it into 32-row dtrsm_ +
//   dgemm_ steps).  Each workgroup owns a strip of 16 columns of A12, keeps
//   it in LDS, and walks L11 in 32-column blocks staged through LDS: solve the
//   32 x 32 diagonal block, then update the rows below with one fma chain.
//
// trsv_persistent: the two solves of PDGETRS (SRC/pdgetrs.f:260-266 for
//   TRANS = 'N', :273-284 for 'T') and of PDLATRS inside PDGECON
//   (SRC/pdgecon.f:342-370) for a few right-hand sides.  Those are
//   latency-bound, so one launch covers the whole triangle: block row b
//   (64 rows) is owned by the workgroup that takes ticket b; it accumulates
//   -T[b, c] X[c] for every finished block c (X[c] read from a mailbox whose
//   words carry the launch's epoch, bounded wait), then solves its 64 x 64
//   diagonal block as four 16 x 16 triangles, a right-hand side in each row of 16
//   lanes, and publishes X[b].
//   Tickets are taken in start order, so a workgroup only ever waits on
//   workgroups that are already running.  The transposed solves read the
//   off-diagonal block by columns (lane = column of the stored triangle,
//   16 consecutive elements of that column per wave).
#include "sla_common.h"
#include "sla_kernels.h"

#include <algorithm>
#include <cstddef>
#include <type_traits>

namespace sla {

namespace {

typedef double bd4_t __attribute__((ext_vector_type(4)));
typedef float bf4_t __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ auto mfma16x4(T a, T b, typename std::conditional<sizeof(T) == 8, bd4_t,
                                                                            bf4_t>::type c)
{
    if constexpr (sizeof(T) == 8) return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// row of accumulator element r of lane (lr, lk) within a 16 x 16 tile
template <typename T>
__device__ __forceinline__ int mfma_row(int lk, int r)
{
    return sizeof(T) == 8 ? lk + 4 * r : 4 * lk + r;
}

constexpr int TS_CW = 16, TS_KB = 32, TS_MAXM = 256;

template <typename T>
__global__ __launch_bounds__(256) void trsm_llnu_strip_kernel(int m, int n, const T *__restrict__ L,
                                                              int ldl, T *__restrict__ B, int ldb)
{
    __shared__ T Bs[TS_MAXM][TS_CW + 1];
    __shared__ T Ls[TS_MAXM][TS_KB + 1];
    const int c0 = blockIdx.x * TS_CW, tid = threadIdx.x;
    const int c = tid % TS_CW, rg = tid / TS_CW;  // 16 row groups
    for (int idx = tid; idx < m * TS_CW; idx += 256) {
        const int r = idx % m, cc = idx / m;
        Bs[r][cc] = (c0 + cc < n) ? B[r + (size_t)(c0 + cc) * ldb] : T(0);
    }
    for (int kb = 0; kb < m; kb += TS_KB) {
        const int kbb = min(TS_KB, m - kb), rows = m - kb;
        __syncthreads();  // previous block's readers of Ls are done
        for (int idx = tid; idx < rows * kbb; idx += 256) {
            const int r = idx % rows, k = idx / rows;
            Ls[r][k] = L[(size_t)(kb + r) + (size_t)(kb + k) * ldl];
        }
        __syncthreads();
        for (int i = 0; i < kbb; i++) {
            const T x = Bs[kb + i][c];
            for (int r = i + 1 + rg; r < kbb; r += 16) Bs[kb + r][c] = fma(-Ls[r][i], x, Bs[kb + r][c]);
            __syncthreads();
        }
        for (int r = kbb + rg; r < rows; r += 16) {
            T acc = Bs[kb + r][c];
            for (int k = 0; k < kbb; k++) acc = fma(-Ls[r][k], Bs[kb + k][c], acc);
            Bs[kb + r][c] = acc;
        }
    }
    __syncthreads();
    for (int idx = tid; idx < m * TS_CW; idx += 256) {
        const int r = idx % m, cc = idx / m;
        if (c0 + cc < n) B[r + (size_t)(c0 + cc) * ldb] = Bs[r][cc];
    }
}

// m <= 32 rows: the solves between two leaves of a panel.  One wave takes 16
// columns, the four lanes of a quad one of them, lane q rows q, q + 4, ..: a
// step is one DPP move of the solved value and at most eight products a lane
// with L's column from LDS.  The same products in the same order as above, in
// 13 KB of LDS and one wave instead of 102 KB and four.
constexpr int T32_NC = 16;

template <int K, typename T>
__device__ __forceinline__ void t32_steps(T (&b)[8], const T (*Ls)[33], int q)
{
    if constexpr (K < 31) {
        const T x = quad_lane<K % 4>(b[K / 4]);
        const T own = fma(-Ls[K][K / 4 * 4 + q], x, b[K / 4]);
        b[K / 4] = q > K % 4 ? own : b[K / 4];
#pragma unroll
        for (int i = K / 4 + 1; i < 8; i++) b[i] = fma(-Ls[K][4 * i + q], x, b[i]);
        t32_steps<K + 1>(b, Ls, q);
    }
}

template <typename T>
__global__ __launch_bounds__(64) void trsm_llnu32_kernel(int m, int n, const T *__restrict__ L,
                                                         int ldl, T *__restrict__ B, int ldb)
{
    __shared__ T Ls[32][33];  // column k of L in row k, zeros outside the triangle
    __shared__ T Bs[T32_NC][33];
    const int c0 = blockIdx.x * T32_NC, lane = threadIdx.x, r = lane & 31, h = lane >> 5;
    const int c = lane >> 2, q = lane & 3;
#pragma unroll
    for (int k = 0; k < 32; k += 2) {
        const int kk = k + h;
        Ls[kk][r] = (r < m && kk < r) ? L[(size_t)r + (size_t)kk * ldl] : T(0);
    }
#pragma unroll
    for (int k = 0; k < T32_NC; k += 2) {
        const int cc = k + h;
        Bs[cc][r] = (r < m && c0 + cc < n) ? B[(size_t)r + (size_t)(c0 + cc) * ldb] : T(0);
    }
    __syncthreads();
    T b[8];
#pragma unroll
    for (int i = 0; i < 8; i++) b[i] = Bs[c][4 * i + q];
    t32_steps<0>(b, Ls, q);
#pragma unroll
    for (int i = 0; i < 8; i++) Bs[c][4 * i + q] = b[i];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < T32_NC; k += 2) {
        const int cc = k + h;
        if (r < m && c0 + cc < n) B[(size_t)r + (size_t)(c0 + cc) * ldb] = Bs[cc][r];
    }
}

// ---------------------------------------------------------------------------
constexpr int TV_BS = 64, TV_NR = 16, TV_PART = TV_BS / 4;

// The stored matrix holds L (unit lower, below the diagonal) and U (upper).
//   !TRANS,  FORWARD: X = L^{-1} X        !TRANS, !FORWARD: X = U^{-1} X
//    TRANS,  FORWARD: X = U^{-T} X         TRANS, !FORWARD: X = L^{-T} X
// A non-unit diagonal is applied as a product with its reciprocals, computed
// before any wait so they stay off the dependency chain.  X is n x nrhs
// (nrhs <= NR <= 16) with leading dimension ldx; the matrix is n x n.
// TA: storage type of the triangle; T: type of X and of the arithmetic (a
// FP32 factorization may be applied in FP64, as GMRES-IR's preconditioner).
//
// Hand-off between blocks: a solved block publishes its values in a mailbox
// of 64-bit words, each holding 32 bits of a value and the launch's epoch in
// the upper half (a double takes two words), written with agent-coherent
// stores.  A waiting workgroup polls the words themselves until every one
// carries the epoch -- one memory round trip from producer to consumer, no
// separate flag and no store drain.  Stale words of earlier launches hold older
// epochs; the mailbox is zeroed when allocated.  The next off-diagonal block of
// the triangle is loaded into registers before the wait, so the matrix read
// stays off the chain.
//
// Bound: the chain of n / 64 blocks, each a mailbox round trip (about 1.3 us),
// a 64 x 64 product and the 64 steps of the diagonal block.  So all four waves
// poll (a wave has at most four columns, not sixteen), and look at the abort
// flag and the clock every 16th time only: the answer costs a trip of its own.
// Two to sixteen right-hand sides go through the matrix cores, which takes the
// product's reads of X from LDS down to one per 16 rows.  The diagonal block is
// solved as four 16 x 16 triangles with one column in each row of 16 lanes, the
// solved value passed on by a DPP move (4 cycles; a lane read through a scalar
// register, with its hazards, took about twice as long) and every column of a
// group of 16 at once, where one wave used to step through them in turn.
// L and U solve together, n = 16384, us, before -> this: one right-hand side
// 2027 -> 1863, four 3827 -> 2134, sixteen 12379 -> 2618; n = 1024: 148 -> 139,
// 263 -> 153, 810 -> 182; n = 100: 33 -> 32, -, 93 -> 37.
template <typename T>
__device__ __forceinline__ uint32_t tv_half(T v, int w)
{
    if constexpr (sizeof(T) == 8) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        return w ? (uint32_t)(u >> 32) : (uint32_t)u;
    } else {
        return __builtin_bit_cast(uint32_t, v);
    }
}

template <typename T>
__device__ __forceinline__ T tv_join(uint32_t lo, uint32_t hi)
{
    if constexpr (sizeof(T) == 8) {
        return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
    } else {
        (void)hi;
        return __builtin_bit_cast(T, lo);
    }
}

// Steps of a 16 x 16 triangle: lane l holds row l of b[0], and in b[1] .. b[3] what
// the solved values take from a row each of the triangles after it (summed apart:
// one rounding of their size a triangle, not sixteen); e[q][k (TV_BS + 1)] is
// column k of those rows, rd the reciprocals of a non-unit diagonal.  Lane l's
// solved value goes to x.  (Lanes already solved go on subtracting; only x counts.)
// The chain of a step is a product, a DPP move and an fma; the other rows' are off
// it.
template <int S, bool FORWARD, bool UNIT, typename T>
__device__ __forceinline__ void tv_steps(T (&b)[4], T &x, const T *const (&e)[4], const T *rd, int l)
{
    if constexpr (S < 16) {
        constexpr int K = FORWARD ? S : 15 - S;
        const T v = row_lane<K>(UNIT ? b[0] : b[0] * rd[K]);
        x = l == K ? v : x;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = fma(-e[q][K * (TV_BS + 1)], v, b[q]);
        tv_steps<S + 1, FORWARD, UNIT>(b, x, e, rd, l);
    }
}

template <typename TA, typename T, bool FORWARD, bool TRANS, int NR>
__global__ __launch_bounds__(256) void trsv_persistent_kernel(
    int n, int nrhs, const TA *__restrict__ A, int lda, T *X, int ldx, int *ticket,
    uint64_t *mail, unsigned epoch, int *abort_flag, uint64_t spin_limit)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, bd4_t, bf4_t>::type;
    constexpr int WPV = sizeof(T) / 4;  // mailbox words per value
    constexpr bool MF = NR > 1;         // products on MFMA: wave w has rows 16 w ..
    constexpr bool UNIT = (FORWARD != TRANS);  // L and L^T have a unit diagonal
    constexpr int NC = MF ? 16 : 1;     // columns of the LDS arrays
    __shared__ int s_b, s_abort[2];
    __shared__ T Xs[2][TV_BS][NC];
    __shared__ T Ys[NC][TV_BS + 1];
    __shared__ T Part[MF ? 1 : 4][TV_BS];
    __shared__ T Es[TV_BS][TV_BS + 1];  // diagonal block, column k of op(T) in row k
    __shared__ T rd[TV_BS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int nblk = ceil_div(n, TV_BS);

    if (tid == 0) s_b = atomicAdd(ticket, 1);
    if (tid < 2) s_abort[tid] = 0;
    for (int i = tid; i < 2 * TV_BS * NC; i += 256) (&Xs[0][0][0])[i] = T(0);
    __syncthreads();
    const int t = s_b;
    if (t >= nblk) return;
    const int b = FORWARD ? t : nblk - 1 - t;
    const int rb = b * TV_BS, rows = min(TV_BS, n - rb);
    // mailbox word (block c, column j, half w, row r)
    auto mbox = [&](int c, int j, int w, int r) -> uint64_t * {
        return mail + ((((size_t)c * NR + j) * WPV + w) * TV_BS + r);
    };

    // The diagonal block, its reciprocals and the right-hand sides before any
    // wait: they do not depend on other blocks.
    for (int idx = tid; idx < TV_BS * TV_BS; idx += 256) {
        const int r = idx % TV_BS, k = idx / TV_BS;  // stored element (r, k)
        const T x = (r < rows && k < rows) ? (T)A[(size_t)(rb + r) + (size_t)(rb + k) * lda] : T(0);
        if (TRANS) Es[r][k] = x;
        else Es[k][r] = x;
    }
    if (!UNIT && tid < TV_BS) rd[tid] = tid < rows ? T(1) / (T)A[(size_t)(rb + tid) * (lda + 1)] : T(1);
    // MF: element r of the lane is row 16 wave + mfma_row(lk, r), column lr;
    // else thread (wave 0, lane) has row lane
    T rhs[MF ? 4 : 1];
#pragma unroll
    for (int r = 0; r < (MF ? 4 : 1); r++) {
        const int row = MF ? 16 * wave + mfma_row<T>(lk, r) : lane, col = MF ? lr : 0;
        rhs[r] = (row < rows && col < nrhs) ? X[(size_t)(rb + row) + (size_t)col * ldx] : T(0);
    }

    // A 64 x 64 block of op(T) right of (left of) the diagonal block, 16 elements
    // a thread.  MF: row 16 wave + lr, k = 16 lk ..; else row lane, k = 16 wave ..
    const int prow = MF ? 16 * wave + lr : lane, pk = 16 * (MF ? lk : wave);
    TA a[TV_PART];
    auto load_block = [&](int s) {
        const int c = FORWARD ? s : nblk - 1 - s;
        const int cb = c * TV_BS, crows = min(TV_BS, n - cb);
        const TA *Ar = TRANS ? A + (size_t)cb + (size_t)(rb + prow) * lda
                             : A + (size_t)(rb + prow) + (size_t)cb * lda;
        const size_t kstride = TRANS ? 1 : (size_t)lda;
#pragma unroll
        for (int kk = 0; kk < TV_PART; kk++)
            a[kk] = (prow < rows && pk + kk < crows) ? Ar[(size_t)(pk + kk) * kstride] : TA(0);
    };
    if (t > 0) load_block(0);

    // four sums of a quarter of the terms each: their rounding errors are half
    // those of one long sum
    acc_t acc[4] = {};
    T part = T(0);
    // Contributions of the solved blocks, in dependency order.  All threads poll:
    // row lane of columns wave, wave + 4, ..; Xs and s_abort alternate, so one
    // barrier a block is enough.
    for (int s = 0; s < t; s++) {
        const int c = FORWARD ? s : nblk - 1 - s, sb = s & 1;
        const int crows = min(TV_BS, n - c * TV_BS);
        constexpr int JP = (NR + 3) / 4;  // columns a thread polls
        if (lane < crows && wave < nrhs) {
            const uint64_t t0 = wall_clock64();
            unsigned it = 0;
            for (;;) {
                uint64_t got[JP][WPV];
                bool ok = true;
#pragma unroll
                for (int i = 0; i < JP; i++)
#pragma unroll
                    for (int w = 0; w < WPV; w++)
                        got[i][w] = __hip_atomic_load(mbox(c, min(wave + 4 * i, nrhs - 1), w, lane),
                                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int i = 0; i < JP; i++)
#pragma unroll
                    for (int w = 0; w < WPV; w++) ok = ok && (uint32_t)(got[i][w] >> 32) == epoch;
                if (ok) {
#pragma unroll
                    for (int i = 0; i < JP; i++)
                        if (wave + 4 * i < nrhs)
                            Xs[sb][lane][wave + 4 * i] =
                                tv_join<T>((uint32_t)got[i][0], (uint32_t)got[i][WPV - 1]);
                    break;
                }
                // the flag and the clock only now and then: the next poll waits
                // for their answer
                if ((++it & 15u) == 0) {
                    if (__hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                        s_abort[sb] = 1;
                        break;
                    }
                    if (wall_clock64() - t0 > spin_limit) {
                        __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        s_abort[sb] = 1;
                        break;
                    }
                }
                // Workgroups far behind the chain poll less often.  The transposed solves
                // read down columns, which is slow enough at large n for the others'
                // polls to be in the way (one right-hand side, n = 28000, U^T and L^T
                // together: 5.28 ms with 16, 5.12 so; n = 4096 539, 526 us; the same in
                // the other two, n = 4096: 542, 545 us).
                if (TRANS && t - s > 32) __builtin_amdgcn_s_sleep(127);
                else if (t - s > 4) __builtin_amdgcn_s_sleep(16);
            }
        }
        __syncthreads();
        if (s_abort[sb]) return;  // the whole workgroup leaves together
        if constexpr (MF) {
            T xb[TV_PART];
#pragma unroll
            for (int kk = 0; kk < TV_PART; kk++) xb[kk] = Xs[sb][pk + kk][lr];
#pragma unroll
            for (int kk = 0; kk < TV_PART; kk++)
                acc[kk & 3] = mfma16x4<T>((T)a[kk], xb[kk], acc[kk & 3]);
        } else {
#pragma unroll
            for (int kk = 0; kk < TV_PART; kk++) part = fma((T)a[kk], Xs[sb][pk + kk][0], part);
        }
        if (s + 1 < t) load_block(s + 1);
    }
    if constexpr (MF) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            Ys[lr][16 * wave + mfma_row<T>(lk, r)] =
                rhs[r] - ((acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]));
        __syncthreads();
    } else {
        Part[wave][lane] = part;
        __syncthreads();
        if (wave == 0)
            Ys[0][lane] = rhs[0] - (((Part[0][lane] + Part[1][lane]) + Part[2][lane]) + Part[3][lane]);
        __syncthreads();
    }

    // The diagonal block: column j of the right-hand sides in a row of 16 lanes,
    // lane l rows 16 i + l; four 16 x 16 triangles, each solved value going on to
    // the rows below (above) its triangle at once.
    const int j = 4 * wave + lk;
    if (4 * wave < nrhs) {
        const T *y = Ys[MF ? j : 0];
        const uint64_t tag = (uint64_t)epoch << 32;
        T yy[4];  // the rows of the current triangle, then those after it
#pragma unroll
        for (int i = 0; i < 4; i++) yy[i] = y[16 * (FORWARD ? i : 3 - i) + lr];
        auto triangle = [&](int i) {
            const int r0 = 16 * (FORWARD ? i : 3 - i);
            const T *e[4];  // rows r0, and those of yy[1] .. yy[3] (a row of the block if none)
#pragma unroll
            for (int q = 0; q < 4; q++)
                e[q] = &Es[r0][(FORWARD ? min(r0 + 16 * q, TV_BS - 16) : max(r0 - 16 * q, 0)) + lr];
            T x = T(0), bb[4] = {yy[0], T(0), T(0), T(0)};
            tv_steps<0, FORWARD, UNIT>(bb, x, e, rd + r0, lr);
            if (j < nrhs && r0 + lr < rows) {
#pragma unroll
                for (int w = 0; w < WPV; w++)
                    __hip_atomic_store(mbox(b, j, w, r0 + lr), tag | tv_half(x, w),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                X[(size_t)(rb + r0 + lr) + (size_t)j * ldx] = x;
            }
            yy[0] = yy[1] + bb[1], yy[1] = yy[2] + bb[2], yy[2] = yy[3] + bb[3];
        };
        // A short last block has fewer triangles with rows: n = 1, both solves with one
        // right-hand side took 9.8 us with all four, now 6.9; n = 20 11.1, 9.0.
        int first = 0, last = 4;
        if (rows <= TV_BS - 16) {
            const int none = 4 - (rows + 15) / 16;
            if (FORWARD) last -= none;
            else first = none;
            if (!FORWARD)
                for (int i = 0; i < none; i++) yy[0] = yy[1], yy[1] = yy[2], yy[2] = yy[3];
        }
        // A loop of its own for whole blocks: the plain solves are 2 % slower without
        // it, the transposed ones with it (n = 8192, two right-hand sides: 1112 and 1130
        // us, 1122 and 1078), by how the compiler schedules the steps.
        if (!TRANS && rows > TV_BS - 16) {
#pragma unroll 1
            for (int i = 0; i < 4; i++) triangle(i);
        } else {
#pragma unroll 1
            for (int i = first; i < last; i++) triangle(i);
        }
    }
}

// ---------------------------------------------------------------------------
// Block-inverse solves with the factors of a low-precision factorization
// (the corrections of iterative refinement and GMRES-IR's preconditioner).
// The inverses of the 128 x 128 diagonal blocks of L and U are formed once
// per factorization, so a step of the dependency chain is two products with
// blocks already in registers instead of 128 dependent substitution steps:
//   x_b = D_b^{-1} (rhs_b - sum_{c before b} T[b, c] x_c).
constexpr int TB_BS = 128, TB_KH = TB_BS / 2, TB_INV_COLS = 64;

// inv holds plane 0 = the inverses of L's unit-lower diagonal blocks and
// plane 1 = those of U's upper diagonal blocks, FP64, block b at
// inv + (plane * nblk + b) * 128 * 128, column-major (element (r, k) at
// k * 128 + r), zero outside the triangle; rows past n are the identity's.
// Workgroup (b, half, plane): one wave, lane j forms column 64 half + j by
// substitution against e_j in FP64, the block staged in LDS (all lanes read
// the same element: a broadcast) and the column in LDS (each lane its own).
template <typename TA>
__global__ __launch_bounds__(TB_INV_COLS) void trsv_diag_inverse_kernel(int n, const TA *__restrict__ A,
                                                                       int lda, double *__restrict__ inv)
{
    __shared__ TA Ds[TB_BS][TB_BS + 1];
    __shared__ double Xs[TB_BS][TB_INV_COLS];
    const int b = blockIdx.x, half = blockIdx.y, plane = blockIdx.z;
    const int nblk = gridDim.x, rb = b * TB_BS, rows = min(TB_BS, n - rb);
    const int lane = threadIdx.x, j = half * TB_INV_COLS + lane;
    for (int idx = lane; idx < TB_BS * TB_BS; idx += TB_INV_COLS) {
        const int r = idx % TB_BS, k = idx / TB_BS;
        TA v = (r == k) ? TA(1) : TA(0);
        if (r < rows && k < rows) v = A[(size_t)(rb + r) + (size_t)(rb + k) * lda];
        Ds[r][k] = v;
    }
    __syncthreads();
    if (plane == 0) {
        // unit lower: x_i = e_j(i) - sum_{k < i} L(i, k) x_k
        for (int i = 0; i < TB_BS; i++) {
            double s = (i == j) ? 1.0 : 0.0;
            for (int k = 0; k < i; k++) s = fma(-(double)Ds[i][k], Xs[k][lane], s);
            Xs[i][lane] = s;
        }
    } else {
        // upper: x_i = (e_j(i) - sum_{k > i} U(i, k) x_k) / U(i, i)
        for (int i = TB_BS - 1; i >= 0; i--) {
            double s = (i == j) ? 1.0 : 0.0;
            for (int k = i + 1; k < TB_BS; k++) s = fma(-(double)Ds[i][k], Xs[k][lane], s);
            Xs[i][lane] = s / (double)Ds[i][i];
        }
    }
    double *out = inv + ((size_t)plane * nblk + b) * TB_BS * TB_BS + (size_t)j * TB_BS;
    for (int i = 0; i < TB_BS; i++) out[i] = Xs[i][lane];
}

// X <- L^{-1} X (FORWARD) or U^{-1} X for the FP32 factors at A with the
// block inverses at inv (plane 0 / 1), nrhs <= NR <= 16, T the arithmetic.
// Same ticket / epoch-tagged mailbox protocol as trsv_persistent_kernel, with
// 128-row blocks: thread (r, h) = (tid % 128, tid / 128) owns row r and the
// k-half h of every block it multiplies; waves 0 and 1 poll the 128 rows of
// the block they wait for.
template <typename T, bool FORWARD, int NR>
__global__ __launch_bounds__(256) void trsv_blockinv_kernel(
    int n, int nrhs, const float *__restrict__ A, int lda, const double *__restrict__ inv, T *X,
    int ldx, int *ticket, uint64_t *mail, unsigned epoch, int *abort_flag, uint64_t spin_limit)
{
    constexpr int WPV = sizeof(T) / 4;
    __shared__ int s_b, s_abort;
    __shared__ T Xs[TB_BS][NR];
    __shared__ T Ph[2][TB_BS][NR + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = tid % TB_BS, h = tid / TB_BS;
    const int nblk = ceil_div(n, TB_BS);
    if (tid == 0) {
        s_b = atomicAdd(ticket, 1);
        s_abort = 0;
    }
    __syncthreads();
    const int t = s_b;
    if (t >= nblk) return;
    const int b = FORWARD ? t : nblk - 1 - t;
    const int rb = b * TB_BS, rows = min(TB_BS, n - rb);
    auto mbox = [&](int c, int j, int w, int row) -> uint64_t * {
        return mail + ((((size_t)c * NR + j) * WPV + w) * TB_BS + row);
    };

    // the diagonal block's inverse, row r, columns of half h (before any wait)
    T dv[TB_KH];
    {
        const double *Di = inv + ((size_t)(FORWARD ? 0 : 1) * nblk + b) * TB_BS * TB_BS;
#pragma unroll
        for (int kk = 0; kk < TB_KH; kk++) dv[kk] = (T)Di[(size_t)(h * TB_KH + kk) * TB_BS + r];
    }
    T rhs[NR], part[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) {
        rhs[j] = (h == 0 && r < rows && j < nrhs) ? X[(size_t)(rb + r) + (size_t)j * ldx] : T(0);
        part[j] = T(0);
    }
    float a[TB_KH];
    auto load_block = [&](int s) {
        const int c = FORWARD ? s : nblk - 1 - s;
        const int cb = c * TB_BS, crows = min(TB_BS, n - cb);
        const float *Ar = A + (size_t)(rb + r) + (size_t)(cb + h * TB_KH) * lda;
#pragma unroll
        for (int kk = 0; kk < TB_KH; kk++)
            a[kk] = (r < rows && h * TB_KH + kk < crows) ? Ar[(size_t)kk * lda] : 0.f;
    };
    if (t > 0) load_block(0);

    for (int s = 0; s < t; s++) {
        const int c = FORWARD ? s : nblk - 1 - s;
        const int crows = min(TB_BS, n - c * TB_BS);
        if (wave < 2) {
            const int row = wave * 64 + lane;
            uint32_t got[NR][WPV];
            int ab = 0;
            const uint64_t t0 = wall_clock64();
            for (;;) {
                bool ok = true;
                if (row < crows) {
#pragma unroll
                    for (int j = 0; j < NR; j++) {
                        if (j < nrhs) {
#pragma unroll
                            for (int w = 0; w < WPV; w++) {
                                const uint64_t u = __hip_atomic_load(
                                    mbox(c, j, w, row), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                got[j][w] = (uint32_t)u;
                                ok = ok && (uint32_t)(u >> 32) == epoch;
                            }
                        }
                    }
                }
                if (__all(ok)) break;
                if (__hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    ab = 1;
                    break;
                }
                if (wall_clock64() - t0 > spin_limit) {
                    __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ab = 1;
                    break;
                }
                if (t - s > 4) __builtin_amdgcn_s_sleep(16);
                else __builtin_amdgcn_s_sleep(1);
            }
#pragma unroll
            for (int j = 0; j < NR; j++)
                Xs[row][j] = (row < crows && j < nrhs) ? tv_join<T>(got[j][0], got[j][WPV - 1]) : T(0);
            if (ab) s_abort = 1;
        }
        __syncthreads();
        if (s_abort) return;  // the whole workgroup leaves together
#pragma unroll
        for (int kk = 0; kk < TB_KH; kk++) {
            const T av = (T)a[kk];
#pragma unroll
            for (int j = 0; j < NR; j++) part[j] = fma(av, Xs[h * TB_KH + kk][j], part[j]);
        }
        if (s + 1 < t) load_block(s + 1);
        __syncthreads();  // Xs is reused by the next block
    }
    // y = rhs - (part_0 + part_1), then x = D^{-1} y as two half products
#pragma unroll
    for (int j = 0; j < NR; j++) Ph[h][r][j] = part[j];
    __syncthreads();
    if (h == 0) {
#pragma unroll
        for (int j = 0; j < NR; j++) Xs[r][j] = r < rows ? rhs[j] - (Ph[0][r][j] + Ph[1][r][j]) : T(0);
    }
    __syncthreads();
    T q[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) q[j] = T(0);
#pragma unroll
    for (int kk = 0; kk < TB_KH; kk++) {
        const T d = dv[kk];
#pragma unroll
        for (int j = 0; j < NR; j++) q[j] = fma(d, Xs[h * TB_KH + kk][j], q[j]);
    }
#pragma unroll
    for (int j = 0; j < NR; j++) Ph[h][r][j] = q[j];
    __syncthreads();
    if (h == 0 && r < rows) {
        const uint64_t tag = (uint64_t)epoch << 32;
#pragma unroll
        for (int j = 0; j < NR; j++) {
            if (j < nrhs) {
                const T x = Ph[0][r][j] + Ph[1][r][j];
#pragma unroll
                for (int w = 0; w < WPV; w++)
                    __hip_atomic_store(mbox(b, j, w, r), tag | tv_half(x, w), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                X[(size_t)(rb + r) + (size_t)j * ldx] = x;
            }
        }
    }
}

}  // namespace

void trsv_block_inverses(int n, const float *A, int lda, double *inv, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(trsv_diag_inverse_kernel<float>, dim3(ceil_div(n, TB_BS), 2, 2),
                       dim3(TB_INV_COLS), 0, s, n, A, lda, inv);
    SLA_LAUNCH_CHECK();
}

template <typename T>
void trsv_blockinv(bool lower, int n, int nrhs, const float *A, int lda, const double *inv, T *X,
                   int ldx, TrsvWork &tw, hipStream_t s)
{
    if (n <= 0 || nrhs <= 0) return;
    if (nrhs > TV_NR) throw std::logic_error("trsv_blockinv: at most 16 right-hand sides per call");
    const int nblk = ceil_div(n, TB_BS);
    if ((size_t)nblk * TB_BS * TV_NR * 2 > tw.mail_words)
        throw std::logic_error("trsv_blockinv: mailbox too small for this order");
    fill_int(tw.ticket, 1, 0, s);
    const int epoch = ++tw.epoch;
#define SLA_TBI(FW, NRV)                                                                          \
    hipLaunchKernelGGL((trsv_blockinv_kernel<T, FW, NRV>), dim3(nblk), dim3(256), 0, s, n, nrhs, \
                       A, lda, inv, X, ldx, tw.ticket, tw.mail, (unsigned)epoch, tw.abort_flag,  \
                       tw.spin_limit)
#define SLA_TBI_NR(FW)                          \
    do {                                        \
        if (nrhs <= 1) SLA_TBI(FW, 1);          \
        else if (nrhs <= 2) SLA_TBI(FW, 2);     \
        else if (nrhs <= 4) SLA_TBI(FW, 4);     \
        else if (nrhs <= 8) SLA_TBI(FW, 8);     \
        else SLA_TBI(FW, 16);                   \
    } while (0)
    if (lower) SLA_TBI_NR(true);
    else SLA_TBI_NR(false);
#undef SLA_TBI_NR
#undef SLA_TBI
    SLA_LAUNCH_CHECK();
}
template void trsv_blockinv<float>(bool, int, int, const float *, int, const double *, float *,
                                   int, TrsvWork &, hipStream_t);
template void trsv_blockinv<double>(bool, int, int, const float *, int, const double *, double *,
                                    int, TrsvWork &, hipStream_t);

template <typename T>
void trsm_llnu(int m, int n, const T *L, int ldl, T *B, int ldb, hipStream_t s)
{
    if (m <= 0 || n <= 0) return;
    if (m > TS_MAXM) throw std::logic_error("trsm_llnu: at most 256 rows per call");
    if (m <= 32) {
        hipLaunchKernelGGL(trsm_llnu32_kernel<T>, dim3(ceil_div(n, T32_NC)), dim3(64), 0, s, m, n, L,
                           ldl, B, ldb);
        SLA_LAUNCH_CHECK();
        return;
    }
    hipLaunchKernelGGL(trsm_llnu_strip_kernel<T>, dim3(ceil_div(n, TS_CW)), dim3(256), 0, s, m, n,
                       L, ldl, B, ldb);
    SLA_LAUNCH_CHECK();
}
template void trsm_llnu<double>(int, int, const double *, int, double *, int, hipStream_t);
template void trsm_llnu<float>(int, int, const float *, int, float *, int, hipStream_t);

// ---------------------------------------------------------------------------
// trsm_llnu_blocked: the same solve for m <= 512 rows in one launch (plus one
// for the inverses, which a second solve with the same L11 reuses), the
// products on MFMA.  L11 is taken in 32-row blocks; the inverse of each unit
// lower 32 x 32 diagonal block is formed by trsm_diag_inv_kernel (thread =
// element, forward substitution against the identity, one barrier per row;
// a block cut by m is completed with the identity).  Each workgroup (8
// waves) owns 16 columns of B, held in LDS, and for block k
//   X_k = inv(L_kk) B_k                     (waves 0, 1: a 16-row tile each)
//   B_i -= L_ik X_k  for the rows below     (16-row tiles, two per wave at a
//                                            time so 16 loads are in flight)
// with v_mfma_f64_16x16x4f64 (FP32: v_mfma_f32_16x16x4f32), L read from
// global memory (L2-resident across the workgroups), X_k from LDS; the next
// block's inverse operands are loaded during the current block's update.
namespace {

constexpr int TB_M = 512, TB_NC = 16, TB_LD = TB_NC + 1;

template <typename T>
__global__ __launch_bounds__(1024) void trsm_diag_inv_kernel(int m, const T *__restrict__ L,
                                                             int ldl, T *__restrict__ inv)
{
    // thread (i, j) holds element (i, j) of the inverse; step k subtracts
    // D_ik x_kj from the rows below k (forward substitution, column-parallel)
    __shared__ T Ds[32][33], Xs[32][33];
    const int b = blockIdx.x, tid = threadIdx.x, i = tid % 32, j = tid / 32, r0 = 32 * b;
    Ds[i][j] = (r0 + i < m && r0 + j < m && i > j) ? L[(size_t)(r0 + i) + (size_t)(r0 + j) * ldl]
                                                  : T(0);
    T x = (i == j) ? T(1) : T(0);
    Xs[i][j] = x;
    for (int k = 0; k < 31; k++) {
        __syncthreads();
        if (i > k) {
            x = fma(-Ds[i][k], Xs[k][j], x);
            if (i == k + 1) Xs[i][j] = x;  // row k + 1 is final
        }
    }
    inv[(size_t)b * 1024 + (size_t)j * 32 + i] = x;
}

// MM: rows at most.  The panel's solves (MM <= 256) run beside the trailing
// update, whose workgroups fill every CU four at a time: 256 threads and a strip
// of MM rows fit where one of them has left, 512 threads with 70 KB of LDS wait
// until a CU is nearly empty (22 us a solve alone, 155 us beside the update).
template <typename T, int MM>
__global__ __launch_bounds__(MM > 256 ? 512 : 256)
__attribute__((amdgpu_waves_per_eu(4))) void trsm_llnu_blocked_kernel(
    int m, int n, const T *__restrict__ L, int ldl, const T *__restrict__ inv, T *__restrict__ B,
    int ldb)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, bd4_t, bf4_t>::type;
    constexpr int TB_T = MM > 256 ? 512 : 256, NW = TB_T / 64;
    __shared__ T Xs[MM][TB_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int c0 = blockIdx.x * TB_NC;
    const int nblk = (m + 31) / 32, m32 = 32 * nblk;
    // B strip into LDS (rows >= m and columns >= n as zeros)
    for (int idx = tid; idx < m32 * TB_NC; idx += TB_T) {
        const int r = idx % m32, c = idx / m32;
        Xs[r][c] = (r < m && c0 + c < n) ? B[(size_t)r + (size_t)(c0 + c) * ldb] : T(0);
    }
    // inverse operands of block 0 (waves 0, 1)
    T iva[8];
    if (wave < 2) {
#pragma unroll
        for (int s = 0; s < 8; s++) iva[s] = inv[(size_t)(4 * s + lk) * 32 + 16 * wave + lr];
    }
    __syncthreads();
    for (int k = 0; k < nblk; k++) {
        const int kr = 32 * k;
        // X_k = inv(L_kk) B_k: waves 0, 1 take rows kr + 16 wave ..
        acc_t d = acc_t{0, 0, 0, 0};
        if (wave < 2) {
#pragma unroll
            for (int s = 0; s < 8; s++) d = mfma16x4<T>(iva[s], Xs[kr + 4 * s + lk][lr], d);
            if (k + 1 < nblk) {  // next block's inverse, in flight during this block's update
                const T *iv = inv + (size_t)(k + 1) * 1024;
#pragma unroll
                for (int s = 0; s < 8; s++) iva[s] = iv[(size_t)(4 * s + lk) * 32 + 16 * wave + lr];
            }
        }
        __syncthreads();  // every read of B_k is done
        if (wave < 2) {
#pragma unroll
            for (int r = 0; r < 4; r++) Xs[kr + 16 * wave + mfma_row<T>(lk, r)][lr] = d[r];
        }
        __syncthreads();  // X_k is final
        const int ntile = (m32 - kr - 32) / 16;  // 16-row tiles below block k
        if (ntile <= 0) break;
        // -X_k as the B operand of every tile of this block
        T xb[8];
#pragma unroll
        for (int s = 0; s < 8; s++) xb[s] = -Xs[kr + 4 * s + lk][lr];
        // tiles t and t + NW together: 16 loads of L in flight per lane
        for (int t = wave; t < ntile; t += 2 * NW) {
            T a[2][8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int row = kr + 32 + 16 * (t + h * NW) + lr;
                const T *lp = L + (size_t)row + (size_t)kr * ldl;
                const bool in = t + h * NW < ntile && row < m;
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const int col = 4 * s + lk;
                    a[h][s] = (in && kr + col < m) ? lp[(size_t)col * ldl] : T(0);
                }
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (t + h * NW >= ntile) break;
                const int r0 = kr + 32 + 16 * (t + h * NW);
                acc_t c;
#pragma unroll
                for (int r = 0; r < 4; r++) c[r] = Xs[r0 + mfma_row<T>(lk, r)][lr];
#pragma unroll
                for (int s = 0; s < 8; s++) c = mfma16x4<T>(a[h][s], xb[s], c);
#pragma unroll
                for (int r = 0; r < 4; r++) Xs[r0 + mfma_row<T>(lk, r)][lr] = c[r];
            }
        }
        __syncthreads();  // block k + 1 is updated
    }
    for (int idx = tid; idx < m * TB_NC; idx += TB_T) {
        const int r = idx % m, c = idx / m;
        if (c0 + c < n) B[(size_t)r + (size_t)(c0 + c) * ldb] = Xs[r][c];
    }
}

// ---------------------------------------------------------------------------
// trsm_tri: one diagonal block (at most 256 rows) of PDGETRS's solves for many
// right-hand sides; the products with the rest of the triangle are GEMMs between
// these launches (trsm_solve).  All four triangles are forward substitutions
// with a lower triangle E of signed strides: E(i, j) = E[i rs + j cs], row i of X
// at X[i xs]; U and L^T run from their last row up, U^T and L^T are read along
// their columns.
//
// A workgroup of four waves keeps 16 columns of X in LDS and walks E in 32-row
// blocks: one wave solves the diagonal block by substitution (a quad of lanes a
// column, as trsm_llnu32_kernel; a non-unit diagonal as products with its
// reciprocals), then all waves subtract E_ik X_k from the rows below on MFMA, 16
// rows a tile, the first tile's E loaded before the solve it waits for.  Bound
// by that chain, about 6 us per 32 rows, and not by the work: with the GEMMs
// n = 5000 and 400 right-hand sides take 3.4 ms where sixteen at a time through
// trsv_persistent took 96 ms.
constexpr int TT_M = 256, TT_T = 256;

template <int K, bool UNIT, typename T>
__device__ __forceinline__ void tri_steps(T (&b)[8], const T (*Es)[33], const T *rd, int q)
{
    if constexpr (K < 32) {
        if (!UNIT) {
            const T x = b[K / 4] * rd[K];
            b[K / 4] = q == K % 4 ? x : b[K / 4];
        }
        const T x = quad_lane<K % 4>(b[K / 4]);
        const T own = fma(-Es[K][K / 4 * 4 + q], x, b[K / 4]);
        b[K / 4] = q > K % 4 ? own : b[K / 4];
#pragma unroll
        for (int i = K / 4 + 1; i < 8; i++) b[i] = fma(-Es[K][4 * i + q], x, b[i]);
        tri_steps<K + 1, UNIT>(b, Es, rd, q);
    }
}

template <typename T, bool UNIT>
__global__ __launch_bounds__(TT_T) void trsm_tri_kernel(int m, int n, const T *__restrict__ E,
                                                        ptrdiff_t rs, ptrdiff_t cs,
                                                        T *__restrict__ X, ptrdiff_t xs, size_t ldx)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, bd4_t, bf4_t>::type;
    constexpr int NW = TT_T / 64;
    __shared__ T Xs[TT_M][TB_LD];
    __shared__ T Es[32][33];  // the diagonal block, column k in row k
    __shared__ T rd[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4, c0 = blockIdx.x * TB_NC;
    const int nblk = (m + 31) / 32, m32 = 32 * nblk;
    for (int idx = tid; idx < m32 * TB_NC; idx += TT_T) {
        const int r = idx % m32, c = idx / m32;
        Xs[r][c] = (r < m && c0 + c < n) ? X[r * xs + (size_t)(c0 + c) * ldx] : T(0);
    }
    // the 16 rows of tile t below block k, columns kr .. kr + 31 of E
    auto load_tile = [&](T (&a)[8], int kr, int t, int ntile) {
        const int row = kr + 32 + 16 * t + lr;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int col = kr + 4 * s + lk;
            a[s] = (t < ntile && row < m) ? E[row * rs + col * cs] : T(0);  // col < m: rows follow
        }
    };
    for (int k = 0; k < nblk; k++) {
        const int kr = 32 * k, ntile = (m32 - kr - 32) / 16;
        // (Es: wave 0, its only reader, was done with block k - 1's before the barrier
        // that made X_{k-1} final)
        for (int idx = tid; idx < 1024; idx += TT_T) {
            const int r = idx & 31, c = idx >> 5;
            Es[c][r] = (c < r && kr + r < m) ? E[(kr + r) * rs + (kr + c) * cs] : T(0);
        }
        if (!UNIT && tid < 32) rd[tid] = kr + tid < m ? T(1) / E[(kr + tid) * (rs + cs)] : T(1);
        T a[8];
        load_tile(a, kr, wave, ntile);
        __syncthreads();  // Es, and X_k's last update
        if (wave == 0) {
            const int c = lane >> 2, q = lane & 3;
            T b[8];
#pragma unroll
            for (int i = 0; i < 8; i++) b[i] = Xs[kr + 4 * i + q][c];
            tri_steps<0, UNIT>(b, Es, rd, q);
#pragma unroll
            for (int i = 0; i < 8; i++) Xs[kr + 4 * i + q][c] = b[i];
        }
        __syncthreads();  // X_k is final
        if (ntile <= 0) break;
        T xb[8];
#pragma unroll
        for (int s = 0; s < 8; s++) xb[s] = -Xs[kr + 4 * s + lk][lr];
        for (int t = wave; t < ntile; t += NW) {
            T an[8];
            load_tile(an, kr, t + NW, ntile);
            const int r0 = kr + 32 + 16 * t;
            // summed apart from X, which then takes one rounding a block and not eight
            acc_t c[2] = {};
#pragma unroll
            for (int s = 0; s < 8; s++) c[s & 1] = mfma16x4<T>(a[s], xb[s], c[s & 1]);
#pragma unroll
            for (int r = 0; r < 4; r++) Xs[r0 + mfma_row<T>(lk, r)][lr] += c[0][r] + c[1][r];
#pragma unroll
            for (int s = 0; s < 8; s++) a[s] = an[s];
        }
    }
    for (int idx = tid; idx < m * TB_NC; idx += TT_T) {
        const int r = idx % m, c = idx / m;
        if (c0 + c < n) X[r * xs + (size_t)(c0 + c) * ldx] = Xs[r][c];
    }
}

}  // namespace

// X <- op(T)^{-1} X, n x nrhs: the diagonal blocks in order, each followed by the
// product of its solution with the rest of its block column (row).
void trsm_solve(TrsvOp op, int n, int nrhs, const double *A, int lda, double *X, int ldx,
                hipStream_t s)
{
    if (n <= 0 || nrhs <= 0) return;
    const bool fwd = op == TrsvOp::L || op == TrsvOp::UT;
    const bool trans = op == TrsvOp::UT || op == TrsvOp::LT;
    const ptrdiff_t rs = (fwd ? 1 : -1) * (trans ? (ptrdiff_t)lda : 1);
    const ptrdiff_t cs = (fwd ? 1 : -1) * (trans ? 1 : (ptrdiff_t)lda);
    const int nblk = ceil_div(n, TT_M);
    for (int i = 0; i < nblk; i++) {
        const int k0 = (fwd ? i : nblk - 1 - i) * TT_M, kb = std::min(TT_M, n - k0), k1 = k0 + kb;
        const int first = fwd ? k0 : k1 - 1;  // the block's row 0 as the kernel counts
        const double *E = A + (size_t)first + (size_t)first * lda;
        const dim3 grid(ceil_div(nrhs, TB_NC));
        if (op == TrsvOp::L || op == TrsvOp::LT)
            hipLaunchKernelGGL((trsm_tri_kernel<double, true>), grid, dim3(TT_T), 0, s, kb, nrhs, E,
                               rs, cs, X + first, (ptrdiff_t)(fwd ? 1 : -1), (size_t)ldx);
        else
            hipLaunchKernelGGL((trsm_tri_kernel<double, false>), grid, dim3(TT_T), 0, s, kb, nrhs, E,
                               rs, cs, X + first, (ptrdiff_t)(fwd ? 1 : -1), (size_t)ldx);
        SLA_LAUNCH_CHECK();
        const int r0 = fwd ? k1 : 0, r1 = fwd ? n : k0;  // rows still to be solved
        const double *off = trans ? A + (size_t)k0 + (size_t)r0 * lda : A + (size_t)r0 + (size_t)k0 * lda;
        gemm_tile_sub<double>(trans, r1 - r0, nrhs, kb, off, lda, X + k0, ldx, X + r0, ldx, s, false, 0,
                              false, nullptr, true);
    }
}

template <typename T>
void trsm_llnu_blocked(int m, int n, const T *L, int ldl, T *B, int ldb, T *inv, bool inv_ready,
                       hipStream_t s)
{
    if (m <= 0 || n <= 0) return;
    if (m > TB_M) throw std::logic_error("trsm_llnu_blocked: at most 512 rows per call");
    const int nblk = (m + 31) / 32;
    if (!inv_ready) {
        hipLaunchKernelGGL(trsm_diag_inv_kernel<T>, dim3(nblk), dim3(1024), 0, s, m, L, ldl, inv);
        SLA_LAUNCH_CHECK();
    }
#define SLA_TB(MV, TV)                                                                            \
    hipLaunchKernelGGL((trsm_llnu_blocked_kernel<T, MV>), dim3(ceil_div(n, TB_NC)), dim3(TV), 0, s, \
                       m, n, L, ldl, (const T *)inv, B, ldb)
    if (m <= 64) SLA_TB(64, 256);
    else if (m <= 128) SLA_TB(128, 256);
    else if (m <= 256) SLA_TB(256, 256);
    else SLA_TB(512, 512);
#undef SLA_TB
    SLA_LAUNCH_CHECK();
}
template void trsm_llnu_blocked<double>(int, int, const double *, int, double *, int, double *,
                                        bool, hipStream_t);
template void trsm_llnu_blocked<float>(int, int, const float *, int, float *, int, float *, bool,
                                       hipStream_t);

template <typename TA, typename T>
void trsv_persistent(TrsvOp op, int n, int nrhs, const TA *A, int lda, T *X, int ldx,
                     TrsvWork &tw, hipStream_t s)
{
    if (n <= 0 || nrhs <= 0) return;
    if (nrhs > TV_NR) throw std::logic_error("trsv_persistent: at most 16 right-hand sides per call");
    const int nblk = ceil_div(n, TV_BS);
    if ((size_t)nblk * TV_BS * TV_NR * 2 > tw.mail_words)
        throw std::logic_error("trsv_persistent: mailbox too small for this order");
    fill_int(tw.ticket, 1, 0, s);
    const int epoch = ++tw.epoch;
#define SLA_TRSV(FW, TR, NRV)                                                                  \
    hipLaunchKernelGGL((trsv_persistent_kernel<TA, T, FW, TR, NRV>), dim3(nblk), dim3(256), 0, \
                       s, n, nrhs, A, lda, X, ldx, tw.ticket, tw.mail, (unsigned)epoch,        \
                       tw.abort_flag, tw.spin_limit)
#define SLA_TRSV_NR(FW, TR)                           \
    do {                                              \
        if (nrhs <= 1) SLA_TRSV(FW, TR, 1);           \
        else if (nrhs <= 4) SLA_TRSV(FW, TR, 4);      \
        else SLA_TRSV(FW, TR, 16);                    \
    } while (0)
    switch (op) {
    case TrsvOp::L: SLA_TRSV_NR(true, false); break;
    case TrsvOp::U: SLA_TRSV_NR(false, false); break;
    case TrsvOp::UT: SLA_TRSV_NR(true, true); break;
    case TrsvOp::LT: SLA_TRSV_NR(false, true); break;
    }
#undef SLA_TRSV_NR
#undef SLA_TRSV
    SLA_LAUNCH_CHECK();
}
template void trsv_persistent<double, double>(TrsvOp, int, int, const double *, int, double *, int,
                                              TrsvWork &, hipStream_t);
template void trsv_persistent<float, float>(TrsvOp, int, int, const float *, int, float *, int,
                                            TrsvWork &, hipStream_t);
template void trsv_persistent<float, double>(TrsvOp, int, int, const float *, int, double *, int,
                                             TrsvWork &, hipStream_t);

}  // namespace sla
