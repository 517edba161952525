// batched.hip -- many independent small systems A_s X_s = B_s (n_s <= 1024,
// nrhs_s <= 16, uneven sizes) factored and solved in ONE persistent launch.
//
// Each system follows the LU path of a 1 x 1 grid: partial pivoting with the
// first maximum |a| of each column (IDAMAX), rows interchanged across the
// whole matrix, the pivot column scaled by the reciprocal of the pivot
// (SRC/pdgetf2.f:206-237), a zero pivot recorded as INFO = column and the
// factorization continued (pdgetrf.f:297-302); then PDGETRS's interchanges
// and two triangular solves (pdgetrs.f:255-266), skipped when INFO > 0
// (pdgesv.f:231).
//
// Work distribution: workgroups take systems from a device queue, largest first
// (the host sorts the sizes once), until the queue is empty; every workgroup
// leaves when the ticket passes the batch size.
//
// Factorization, 512 threads, blocked right-looking with blocks of 64 columns, each
// of W-column panels:
//   panel    held in registers, a thread a row (two rows and 8 columns where more
//            than 512 rows are left); a column costs one workgroup barrier
//            (panel_regs);
//   strips   of 16 columns right of a panel or a block: the interchanges, U12 =
//            L11^{-1} A12 in registers, A22 -= L21 U12 on the 16 x 16 x 4 MFMA of the
//            storage precision, the strip of A22 passing through registers once.
//            After a panel they end at the block and all waves share them; after
//            the block a wave takes a strip by itself, with no barrier in between.
//            Columns on the left get their interchanges only, if there are any.
// Bound: small systems by the chain of columns (under 1 us each: search, post,
// barrier, fold, update), large ones by the passes over A22, n / 64 of them, and over
// L21, once a strip, since the systems in flight (512 of n = 512 are 1 GB) do not
// stay in cache.  512 threads and at most 128 registers keep 16 waves on a CU with
// two workgroups, where 256 threads with 196 registers kept eight.  (In scratch are 16
// bytes a lane with FP64 panels of 32 columns, read back once a block, and 28 of the
// FP64 solve, six values a block of 64 rows; none within a panel, strip or triangle.)  Before, A22 was passed over n / W times, the interchanges of a column
// were one after another in memory, U12 and A22 went through LDS with a barrier
// around every 64 x 64 tile, and the search took eighteen lane exchanges.
// Factorization and solve of 512 systems with interchanges, us, that -> strips behind
// every panel -> blocks: FP64 n = 64 273 -> 165 -> 166, 128 601 -> 350 -> 335, 256
// 1918 -> 1329 -> 973, 512 11095 -> 9332 -> 5310; FP32 257 -> 147 -> 147, 559 -> 299 ->
// 292, 1666 -> 870 -> 703, 8764 -> 5849 -> 3468.  2000 FP64 systems of 32 .. 512, the
// factorization: 12.5 -> 6.0 -> 3.9 ms.
//
// The solves, 512 threads: the interchanges as one permutation, then blocks of 64
// rows for all right-hand sides at once: the diagonal block by substitution on 16 x
// 16 triangles, the rows outside it by MFMA in tiles of 16 rows (solve_triangle).
// Bound by the chain of blocks, about 5 us each, for the systems of a CU in turn.
// Before, blocks of 16 rows each waited for their triangle's row from memory, exchanged
// values through LDS permutes and updated by dot products, and one thread composed
// the interchanges.  2000 FP64 systems of 32 .. 512, one to eight right-hand sides:
// 2.05 -> 0.33 ms; 4000 FP32 systems of 8 .. 160: 227 -> 146 us.
#include "sla_common.h"
#include "sla_handle.h"
#include "sla_batched.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>
#include <numeric>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

namespace sla {

namespace {

constexpr int FT = 512, FW = FT / 64;  // threads and waves of a workgroup
constexpr int SOLVE_WGS = 2;           // workgroups a CU of the solves: what fits
constexpr int SC = 16;                 // columns of a strip
constexpr int KB = 64;                 // columns of a block

struct SysDesc {
    int n, nrhs, lda, ldb;
};

// A pointer that was itself loaded from memory has no known address space, and
// its accesses would be flat: no scalar base, and counted among the LDS accesses
// that a barrier waits for.
template <typename T>
using Global = __attribute__((address_space(1))) T;

typedef double bd4_t __attribute__((ext_vector_type(4)));
typedef float bf4_t __attribute__((ext_vector_type(4)));

// A pivot candidate's rank, (hi, lo) compared as one number: 0 for no candidate,
// then a NaN in row j (kept only if nothing is comparable), then |v|.
__device__ __forceinline__ void rank_of(double v, bool act, bool top, uint32_t &hi, uint32_t &lo)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t h = (uint32_t)(u >> 32) & 0x7fffffffu;
    const bool nan = v != v;
    hi = act ? (nan ? (top ? 1u : 0u) : h + 2u) : 0u;
    lo = nan ? 0u : (uint32_t)u;
}
__device__ __forceinline__ void rank_of(float v, bool act, bool top, uint32_t &hi, uint32_t &lo)
{
    hi = act ? (v != v ? (top ? 1u : 0u) : (__builtin_bit_cast(uint32_t, v) & 0x7fffffffu) + 2u) : 0u;
    lo = 0u;
}

// What the interchanges of the columns at kb do: row kb + i receives row src[i],
// and its old contents go to row dst[i].
template <int W>
struct Moves {
    int src[W], dst[W];
    int any;
};

// LDS of a factorization.  Per column parity: every wave's candidate row with the
// reciprocal of its pivot, its rank and position.
template <typename T, int W>
struct FactorLds {
    alignas(16) T rows[2][FW][W];
    T rcp[2][FW];
    uint32_t hi[2][FW], lo[2][FW];
    int pos[2][FW];
    T L11[W][W + 1];             // column k of the panel's unit lower triangle in row k
    T Lb[KB][KB + 1];            // and of the block's
    T U[FW][16][SC + 1];         // 16 rows of a wave's strip of U12
    int from[BATCHED_NMAX];      // the row that the block's panels moved to each position
    Moves<W> pm;                 // the panel's interchanges
    Moves<KB> bm;                // and the block's
};

// Panel columns kb .. kb + w - 1 of rows kb .. n - 1 held in registers while they
// are factored: thread t holds rows kb + t + 512 q (q < RPT).  Rows stay with
// their thread and carry their position.  Per column j: the wave's first largest
// |a| among the positions >= j (its leading 32 bits decide unless they are
// shared), the owner posts its row and its reciprocal, ONE barrier, every wave
// folds the posts in the same order, the rows below are scaled by the reciprocal
// and updated with the pivot row.  The posts alternate by column parity, so no
// second barrier is needed.  The interchanges reach the other columns in the
// strips that follow, from src and dst.
template <typename T, int W, int RPT, int WL>
__device__ __forceinline__ void panel_regs(int n, int kb, int w, bool first, Global<T> *a, int lda, Global<int> *piv,
                                           int &info, FactorLds<T, WL> &sl)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nw = min(FW, (n - kb + 63) / 64);  // waves that hold rows
    T v[RPT][W];
    int pos[RPT], from[RPT];  // from: the row at the block's start
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int r = kb + tid + FT * q;
        pos[q] = r < n ? r : -1;
        from[q] = r < n && !first ? sl.from[r] : r;
#pragma unroll
        for (int c = 0; c < W; c++)
            v[q][c] = (r < n && c < w) ? (a + (size_t)(kb + c) * lda)[(unsigned)r] : T(0);
    }
    if (tid == 0) sl.pm.any = 0;
    unsigned nopiv = 0;  // columns without a pivot
#pragma unroll
    for (int jj = 0; jj < W; jj++) {
        if (jj < w) {  // uniform
            const int j = kb + jj, pb = jj & 1;
            if (wave < nw) {
                uint32_t bh, bl;
                int bq = 0, bp = pos[0];
                rank_of(v[0][jj], pos[0] >= j, pos[0] == j, bh, bl);
#pragma unroll
                for (int q = 1; q < RPT; q++) {
                    uint32_t h, l;
                    rank_of(v[q][jj], pos[q] >= j, pos[q] == j, h, l);
                    if (h > bh || (h == bh && (l > bl || (l == bl && pos[q] < bp)))) {
                        bh = h, bl = l, bp = pos[q], bq = q;
                    }
                }
                const uint32_t hm = wave_max(bh);
                uint64_t in = __ballot(bh == hm);
                if ((in & (in - 1)) && hm) {
                    const uint32_t lm = wave_max(bh == hm ? bl : 0u);
                    const bool eq = bh == hm && bl == lm;
                    const uint32_t nm = wave_max(eq ? ~(uint32_t)bp : 0u);
                    in = __ballot(eq && ~(uint32_t)bp == nm);
                }
                if (lane == __builtin_ctzll(in)) {
#pragma unroll
                    for (int c = jj; c < W; c++) {
                        T x = v[0][c];
#pragma unroll
                        for (int q = 1; q < RPT; q++) x = bq == q ? v[q][c] : x;
                        sl.rows[pb][wave][c] = x;
                        if (c == jj) sl.rcp[pb][wave] = T(1) / x;
                    }
                    sl.hi[pb][wave] = bh;
                    sl.lo[pb][wave] = bl;
                    sl.pos[pb][wave] = bp;
                }
            }
            lds_barrier();
            const int i = lane & (FW - 1);
            const uint32_t h = i < nw ? sl.hi[pb][i] : 0u;
            const int wp = i < nw ? sl.pos[pb][i] : 0;
            uint32_t hm = dpp_max<0x121, 0xf>(h);
            hm = dpp_max<0x122, 0xf>(hm);
            hm = dpp_max<0x124, 0xf>(hm);
            uint32_t in = (uint32_t)__ballot(h == hm) & ((1u << FW) - 1u);
            if (in & (in - 1)) {
                const uint32_t l = sl.lo[pb][i];
                const uint32_t lm = wave_max(h == hm ? l : 0u);
                const bool eq = h == hm && l == lm;
                const uint32_t nm = wave_max(eq ? ~(uint32_t)wp : 0u);
                in = (uint32_t)__ballot(eq && ~(uint32_t)wp == nm) & ((1u << FW) - 1u);
            }
            const int fw = __builtin_ctz(in);
            const int p = __builtin_amdgcn_readlane(wp, fw);
            const T *prow = sl.rows[pb][fw];
            const T pv = prow[jj], rcp = sl.rcp[pb][fw];
            const bool nz = pv != T(0);
            if (tid == 0) piv[j] = p + 1;
            if (!nz) nopiv |= 1u << jj;
#pragma unroll
            for (int q = 0; q < RPT; q++) {
                if (nz) pos[q] = pos[q] == p ? j : pos[q] == j ? p : pos[q];
                if (pos[q] > j) {
                    const T l = nz ? v[q][jj] * rcp : v[q][jj];
                    v[q][jj] = l;
#pragma unroll
                    for (int c = jj + 1; c < W; c++) v[q][c] = fma(-l, prow[c], v[q][c]);
                }
            }
        }
    }
    if (nopiv) {
        if (info == 0) info = kb + __builtin_ctz(nopiv) + 1;
        // no rows were interchanged (p != j if row j holds a NaN and others zeros)
        if (tid == 0)
            for (unsigned m = nopiv; m; m &= m - 1) {
                const int j = kb + __builtin_ctz(m);
                piv[j] = j + 1;
            }
    }
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int r = kb + tid + FT * q;
        if (r < n) {
#pragma unroll
            for (int c = 0; c < W; c++)
                if (c < w) (a + (size_t)(kb + c) * lda)[(unsigned)pos[q]] = v[q][c];
            if (pos[q] < kb + w)
#pragma unroll
                for (int c = 0; c < W; c++) sl.L11[c][pos[q] - kb] = v[q][c];
            sl.from[pos[q]] = from[q];
            if (pos[q] < kb + w) sl.pm.src[pos[q] - kb] = r;
            if (r < kb + w) sl.pm.dst[r - kb] = pos[q];
            if (pos[q] != r) sl.pm.any = 1;
        }
    }
    __syncthreads();
}

// b <- L^{-1} b for a column in a quad of lanes, lane q rows 4 i + q.  What 16 solved
// values take from the rows after them is summed apart, in s.
template <int K, int W, typename T, int WL>
__device__ __forceinline__ void unit_steps(T (&b)[W / 4], T (&s)[W / 4], const T (*Es)[WL], int q)
{
    if constexpr (K < W) {
        constexpr int I1 = (K / 16 + 1) * 4 < W / 4 ? (K / 16 + 1) * 4 : W / 4;
        const T x = quad_lane<K % 4>(b[K / 4]);
        const T own = fma(-Es[K][K / 4 * 4 + q], x, b[K / 4]);
        b[K / 4] = q > K % 4 ? own : b[K / 4];
#pragma unroll
        for (int i = K / 4 + 1; i < I1; i++) b[i] = fma(-Es[K][4 * i + q], x, b[i]);
#pragma unroll
        for (int i = I1; i < W / 4; i++) {
            s[i] = K % 16 ? fma(-Es[K][4 * i + q], x, s[i]) : -Es[K][4 * i + q] * x;
            if (K % 16 == 15) b[i] += s[i];
        }
        // or the reads of many steps ahead take the registers
        if (W > 32 && (K < 32 || K % 2)) __builtin_amdgcn_sched_barrier(0);
        unit_steps<K + 1, W>(b, s, Es, q);
    }
}

// One wave takes the 16 columns c0 .. c0 + 15 (those below cend) through the K
// columns at kb (w of them, w = K with UPDATE): their interchanges (loads of rows
// kb .. and of what they displace, then the stores), and with UPDATE U12 =
// L11^{-1} A12 by substitution, a quad of lanes a column, and A22 -= L21 U12 in
// 16-row tiles on MFMA.  With SPLIT nparts waves share the strip: each forms U12, the
// first stores it, and they take the row tiles in turn; all waves of the workgroup
// call it, those without a strip with c0 >= cend.
// The product is formed transposed, so a load or store of A22 covers 16 consecutive
// rows of four columns rather than four of sixteen.  Loads run ahead of the MFMA by
// 32 columns of L21 and by a tile of A22.
// D layouts: f64 16x16x4, element r of lane l = D[l/16 + 4 r][l % 16];
// f32 16x16x4, element r of lane l = D[4 (l/16) + r][l % 16].
template <bool UPDATE, bool SPLIT, int K, typename T, int LD>
__device__ __forceinline__ void strip(int n, int kb, int w, int c0, int cend, Global<T> *a, int lda,
                                      const int *src, const int *dst, bool moved, const T (*Es)[LD],
                                      T (*Us)[SC + 1], int part, int nparts)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, bd4_t, bf4_t>::type;
    constexpr int NI = K / 4, UR = K < 16 ? K : 16;  // rows of U12 that change layout at once
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // else a kernel's worth of offsets is kept, in scratch
    const int lr = lane & 15, lk = lane >> 4;
    T b[NI];
    {
        const int q = lane & 3, c = lane >> 2;
        const bool on = c0 + c < cend;
        // loads are clamped into the matrix, not predicated: what they bring from
        // there stays in rows or columns that are not stored
        Global<T> *x = a + (size_t)min(c0 + c, cend - 1) * lda;
        if (moved) {
            T d[NI];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int k = UPDATE ? 4 * i + q : min(4 * i + q, w - 1);
                b[i] = x[(unsigned)src[k]];
                d[i] = x[kb + k];
            }
            if constexpr (SPLIT) __syncthreads();  // all parts have loaded
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int k = 4 * i + q;
                if (on && k < w && (!SPLIT || part == 0)) {
                    const int to = dst[k];
                    if (to >= kb + w) x[(unsigned)to] = d[i];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) b[i] = x[kb + (UPDATE ? 4 * i + q : min(4 * i + q, w - 1))];
        }
        if constexpr (SPLIT) __syncthreads();  // all have loaded; rows of other parts' tiles
        if constexpr (UPDATE) {
            T sum[NI];
            unit_steps<0, K>(b, sum, Es, q);
        }
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (on && 4 * i + q < w && (!SPLIT || part == 0)) x[kb + 4 * i + q] = b[i];
    }
    if constexpr (UPDATE) {
        const int r0 = kb + K, ntile = c0 < cend ? (n - r0 + 15) / 16 : 0;
        if (SPLIT && part >= ntile) return;
        // b <- the B operand, row 4 s + lk of column lr
#pragma unroll
        for (int g = 0; g < K / UR; g++) {
#pragma unroll
            for (int i = 0; i < UR / 4; i++) Us[4 * i + (lane & 3)][lane >> 2] = b[g * UR / 4 + i];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < UR / 4; s++) b[g * UR / 4 + s] = Us[4 * s + lk][lr];
            __builtin_amdgcn_wave_barrier();
        }
        const int cc = c0 + (sizeof(T) == 8 ? lk : 4 * lk);
        constexpr int CS = sizeof(T) == 8 ? 4 : 1;  // columns between a lane's elements
        const Global<T> *L = a + (size_t)(kb + lk) * lda;
        Global<T> *C[4];
#pragma unroll
        for (int r = 0; r < 4; r++) C[r] = a + (size_t)min(cc + CS * r, cend - 1) * lda;
        constexpr int NH = NI > 8 ? 8 : NI, H = NI / NH;  // loads of L21 in H pieces
        T l[2][NH], v[4];
        auto load_l = [&](T(&l)[NH], int t, int h) {
            const Global<T> *Lt = L + min(r0 + lr + 16 * t, n - 1);
            size_t ld = lda;
            asm("" : "+s"(ld));  // else sixteen column addresses are kept, in scratch
#pragma unroll
            for (int s = 0; s < NH; s++) l[s] = Lt[(size_t)(4 * (h * NH + s)) * ld];
        };
        auto load_c = [&](T(&v)[4], int t) {
            const int row = min(r0 + lr + 16 * t, n - 1);
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = C[r][row];
        };
        // the sums of 16 products are formed apart, or a block's rounding errors grow
        // above those of as many panels
        auto mm = [&](acc_t(&acc)[NH > 4 ? 2 : 1], const T(&l)[NH], int h) {
#pragma unroll
            for (int s = 0; s < NH; s++) {
                acc_t &c = acc[s / 4];
                if constexpr (sizeof(T) == 8)
                    c = __builtin_amdgcn_mfma_f64_16x16x4f64(b[h * NH + s], l[s], c, 0, 0, 0);
                else
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(b[h * NH + s], l[s], c, 0, 0, 0);
            }
        };
        auto take = [&](T(&v)[4], const acc_t(&acc)[NH > 4 ? 2 : 1]) {
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] -= NH > 4 ? acc[0][r] + acc[NH > 4][r] : acc[0][r];
        };
        load_l(l[0], part, 0);
        if constexpr (H == 1) load_c(v, part);
        for (int t = part; t < ntile; t += nparts) {
            T vn[4];
            acc_t acc[NH > 4 ? 2 : 1] = {};
            if constexpr (H == 2) {
                load_c(v, t);
                load_l(l[1], t, 1);
                mm(acc, l[0], 0);
                load_l(l[0], t + nparts, 0);
                acc_t acc2[2] = {};
                mm(acc2, l[1], 1);
                take(v, acc);
                take(v, acc2);
            } else {
                load_l(l[1], t + nparts, 0);
                load_c(vn, t + nparts);
                mm(acc, l[0], 0);
                take(v, acc);
#pragma unroll
                for (int s = 0; s < NH; s++) l[0][s] = l[1][s];
            }
            const bool ok = r0 + lr + 16 * t < n;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (ok && cc + CS * r < cend) C[r][r0 + lr + 16 * t] = v[r];
                if constexpr (H == 1) v[r] = vn[r];
            }
        }
    }
}

// The panel at kp of the block kb .. ce - 1 and its strips inside the block; returns
// its width.
template <int W, int RPT, typename T, int WL>
__device__ __forceinline__ int inner_step(int n, int kb, int kp, int ce, Global<T> *a, int lda,
                                          Global<int> *piv, int &info, FactorLds<T, WL> &sl)
{
    const int wave = threadIdx.x >> 6, w = min(W, ce - kp);
    panel_regs<T, W, RPT>(n, kp, w, kp == kb, a, lda, piv, info, sl);
    const int ns = (ce - kp - w + SC - 1) / SC;
    if (ns > 0) {
        const int nparts = FW / ns, si = wave / nparts;
        strip<true, true, W>(n, kp, w, si < ns ? kp + w + SC * si : ce, ce, a, lda, sl.pm.src,
                             sl.pm.dst, sl.pm.any, (const T(*)[WL + 1])sl.L11, sl.U[wave], wave % nparts, nparts);
    }
    if (sl.pm.any)
        for (int c0 = kb + SC * wave; c0 < kp; c0 += SC * FW)
            strip<false, false, W>(n, kp, w, c0, kp, a, lda, sl.pm.src, sl.pm.dst,
                                   true,
                                   (const T(*)[WL + 1])sl.L11, sl.U[wave], 0, 1);
    __syncthreads();  // the block's columns are final before the next panel, sl free
    return w;
}

// P A = L U in place by blocks of 64 columns: panels of W columns (of 8 where more
// than 512 rows are left and a thread keeps two: that fits the registers) and their
// strips inside the block, then the block's strips outside.
template <typename T, int W>
__device__ __forceinline__ void factor_system(int n, Global<T> *a, int lda, Global<int> *piv, int &info,
                              FactorLds<T, W> &sl)
{
    const int tid = threadIdx.x, wave = tid >> 6;
    for (int kb = 0; kb < n; kb += KB) {
        const int wb = min(KB, n - kb), ce = kb + wb;
        for (int kp = kb; kp < ce;) {
            if (n - kp > FT) kp += inner_step<8, 2>(n, kb, kp, ce, a, lda, piv, info, sl);
            else kp += inner_step<W, 1>(n, kb, kp, ce, a, lda, piv, info, sl);
        }
        if (kb == 0 && ce == n) break;
        if (tid == 0) sl.bm.any = 0;
        for (int i = tid; i < KB * KB; i += FT) {
            const int r = i % KB, k = i / KB;
            sl.Lb[k][r] = r < wb && k < wb ? a[(size_t)(kb + r) + (size_t)(kb + k) * lda] : T(0);
        }
        __syncthreads();
        for (int r = kb + tid; r < n; r += FT) {
            const int from = sl.from[r];
            if (r < ce) sl.bm.src[r - kb] = from;
            if (from < ce) sl.bm.dst[from - kb] = r;
            if (from != r) sl.bm.any = 1;
        }
        __syncthreads();
        for (int c0 = ce + SC * wave; c0 < n; c0 += SC * FW)
            strip<true, false, KB>(n, kb, wb, c0, n, a, lda, sl.bm.src, sl.bm.dst, sl.bm.any,
                                   (const T(*)[KB + 1])sl.Lb, sl.U[wave], 0, 1);
        if (sl.bm.any)
            for (int c0 = SC * (FW - 1 - wave); c0 < kb; c0 += SC * FW)
                strip<false, false, KB>(n, kb, wb, c0, kb, a, lda, sl.bm.src, sl.bm.dst, true,
                                        (const T(*)[KB + 1])sl.Lb, sl.U[wave], 0, 1);
        __syncthreads();  // the columns are final before the next panel, sl free
    }
}

// LDS of a solve.
template <typename T>
struct SolveLds {
    T Es[KB][KB + 1];  // the diagonal block, column k in row k
    T Xs[KB][SC + 1];  // its solution
    T rd[KB];          // reciprocals of U's diagonal
    alignas(16) int piv[BATCHED_NMAX];
    int moved;
};

// Steps of a 16 x 16 triangle, top down (L, unit) or bottom up (U): lane l of a row
// of 16 lanes holds row l of b[0], and in b[1] .. b[3] what the solved values take
// from a row each of the triangles after it; e[i][k (KB + 1)] is column k of those
// rows.  A
// quotient is the product with the reciprocal and one correction by its residual;
// where that is not finite it is divided out.
template <int S, bool FWD, typename T>
__device__ __forceinline__ void solve_steps(T (&b)[4], T &x, const T *const (&e)[4], const T *rd, int l)
{
    if constexpr (S < 16) {
        constexpr int K = FWD ? S : 15 - S;
        T v = b[0];
        if (!FWD) {
            const T d = e[0][K * (KB + 1) + K - l], r = rd[K], y = v * r;
            v = fma(fma(-d, y, v), r, y);
            if (!(fabs(v) <= std::numeric_limits<T>::max())) v = b[0] / d;
        }
        v = row_lane<K>(v);
        x = l == K ? v : x;
#pragma unroll
        for (int i = 0; i < 4; i++) b[i] = fma(-e[i][K * (KB + 1)], v, b[i]);
        solve_steps<S + 1, FWD>(b, x, e, rd, l);
    }
}

// X <- L^{-1} X (FWD) or U^{-1} X for all nrhs <= 16 columns at once, right-looking in
// blocks of 64 rows: the diagonal block as four 16 x 16 triangles, a column in each
// row of 16 lanes of waves 0 .. 3, then the rows below (above) in tiles of 16 on MFMA,
// formed transposed like the strips of the factorization.
template <bool FWD, typename T>
__device__ __forceinline__ void solve_triangle(int n, const Global<T> *a, int lda, Global<T> *X, int ldx,
                                               int nrhs, SolveLds<T> &sl)
{
    using acc_t = typename std::conditional<sizeof(T) == 8, bd4_t, bf4_t>::type;
    constexpr int NE = KB * KB / FT, NS = KB / 4;
    constexpr int CS = sizeof(T) == 8 ? 4 : 1;  // columns between a lane's elements
    const int wave = threadIdx.x >> 6, nblk = (n + KB - 1) / KB;
    int lane = threadIdx.x & 63;
    // blocks count from the end they start at: only the last one can be short
    auto first_row = [&](int s) { return FWD ? KB * s : max(n - KB * (s + 1), 0); };
    T en[NE];  // the next diagonal block: row lane, columns wave + 8 i
    auto load_diag = [&](int rb) {
#pragma unroll
        for (int i = 0; i < NE; i++)
            en[i] = a[(size_t)min(rb + lane, n - 1) + (size_t)min(rb + wave + FW * i, n - 1) * lda];
    };
    load_diag(first_row(0));
    for (int s = 0; s < nblk; s++) {
        const int rb = first_row(s), rows = min(KB, FWD ? n - rb : n - KB * s);
        asm volatile("" : "+v"(lane));  // else all offsets of a block are kept, in scratch
        const int lr = lane & 15, lk = lane >> 4;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int k = wave + FW * i;
            const bool in = lane < rows && k < rows;
            sl.Es[k][lane] = in ? en[i] : T(0);
            if (!FWD && lane == k) sl.rd[k] = in ? T(1) / en[i] : T(1);
        }
        const int j = 4 * wave + lk;
        T y[4];
        if (4 * wave < nrhs) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = 16 * (FWD ? i : 3 - i) + lr;
                y[i] = X[(size_t)min(rb + r, n - 1) + (size_t)min(j, nrhs - 1) * ldx];
                y[i] = r < rows ? y[i] : T(0);
            }
        }
        __syncthreads();  // Es
        if (4 * wave < nrhs) {
#pragma unroll 1
            for (int i = 0; i < 4; i++) {
                const int r0 = 16 * (FWD ? i : 3 - i);
                T bb[4] = {y[0], T(0), T(0), T(0)};
                const T *e[4];  // rows r0, and those of bb[1] .. bb[3] (a row of the block if none)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    e[q] = &sl.Es[r0][(FWD ? min(r0 + 16 * q, KB - 16) : max(r0 - 16 * q, 0)) + lr];
                T x = T(0);
                if (r0 < rows) solve_steps<0, FWD>(bb, x, e, sl.rd + r0, lr);
                sl.Xs[r0 + lr][j] = r0 + lr < rows ? x : T(0);
                if (r0 + lr < rows && j < nrhs) X[(size_t)(rb + r0 + lr) + (size_t)j * ldx] = x;
                y[0] = y[1] + bb[1], y[1] = y[2] + bb[2], y[2] = y[3] + bb[3];
            }
        }
        __syncthreads();  // Xs; Es is free
        if (s + 1 == nblk) break;
        const int r0 = FWD ? rb + KB : 0, rend = FWD ? n : rb;
        const int ntile = (rend - r0 + 15) / 16;
        if (wave < ntile) {
            T u[NS];  // columns without a right-hand side hold anything: theirs alone
#pragma unroll
            for (int i = 0; i < NS; i++) u[i] = sl.Xs[4 * i + lk][lr];
            const int cc = sizeof(T) == 8 ? lk : 4 * lk;
            for (int t = wave; t < ntile; t += FW) {
                const int row = r0 + 16 * t + lr, lrow = min(row, rend - 1);
                T l[NS], v[4];
                size_t ld = lda;
                asm("" : "+s"(ld));
                const Global<T> *Lt = a + lrow + (size_t)(rb + lk) * lda;
#pragma unroll
                for (int r = 0; r < 4; r++)
                    v[r] = X[(size_t)lrow + (size_t)min(cc + CS * r, nrhs - 1) * ldx];
#pragma unroll
                for (int i = 0; i < NS; i++) l[i] = Lt[(size_t)(4 * i) * ld];  // a full block
                acc_t acc[4] = {};  // as in the strips
#pragma unroll
                for (int i = 0; i < NS; i++) {
                    acc_t &c = acc[i / 4];
                    if constexpr (sizeof(T) == 8)
                        c = __builtin_amdgcn_mfma_f64_16x16x4f64(u[i], l[i], c, 0, 0, 0);
                    else
                        c = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i], l[i], c, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (row < rend && cc + CS * r < nrhs)
                        X[(size_t)row + (size_t)(cc + CS * r) * ldx] =
                            v[r] - ((acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]));
            }
        }
        load_diag(first_row(s + 1));          // on its way while the stores of X are
        __syncthreads();                     // X, before the next block reads it
    }
}

// X = U^{-1} L^{-1} P B for all nrhs columns of B at once.  The interchanges: each
// thread follows its rows through all of them (n steps on registers, four pivots a
// read of LDS), then the rows move at once.
template <typename T>
__device__ __forceinline__ void solve_all(int n, const Global<T> *a, int lda, const Global<int> *piv,
                                          Global<T> *B, int ldb, int nrhs, SolveLds<T> &sl)
{
    constexpr int RPT = BATCHED_NMAX / FT, NC = 4;
    const int tid = threadIdx.x, n4 = (n + 3) & ~3;
    if (tid == 0) sl.moved = 0;
    __syncthreads();
    for (int i = tid; i < n4; i += FT) {
        const int p = i < n ? piv[i] - 1 : i;
        sl.piv[i] = p;
        if (p != i) sl.moved = 1;
    }
    __syncthreads();
    if (sl.moved) {
        int to[RPT];
#pragma unroll
        for (int q = 0; q < RPT; q++) to[q] = tid + FT * q;
        for (int j = 0; j < n4; j += 4) {
            const int4 p4 = *reinterpret_cast<const int4 *>(&sl.piv[j]);
            const int p[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int q = 0; q < RPT; q++)
                    to[q] = to[q] == j + i ? p[i] : to[q] == p[i] ? j + i : to[q];
        }
        for (int c0 = 0; c0 < nrhs; c0 += NC) {
            T v[RPT][NC];
#pragma unroll
            for (int q = 0; q < RPT; q++)
#pragma unroll
                for (int c = 0; c < NC; c++)
                    v[q][c] = B[(size_t)min(tid + FT * q, n - 1) + (size_t)min(c0 + c, nrhs - 1) * ldb];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < RPT; q++)
#pragma unroll
                for (int c = 0; c < NC; c++)
                    if (tid + FT * q < n && c0 + c < nrhs)
                        B[(size_t)to[q] + (size_t)(c0 + c) * ldb] = v[q][c];
        }
        __syncthreads();
    }
    solve_triangle<true>(n, a, lda, B, ldb, nrhs, sl);
    solve_triangle<false>(n, a, lda, B, ldb, nrhs, sl);
}

template <typename T, int W>
__global__ __launch_bounds__(FT) __attribute__((amdgpu_waves_per_eu(4))) void gesv_batched_kernel(
    int batch, const int *__restrict__ order, const SysDesc *__restrict__ desc,
    T *const *__restrict__ A, int *const *__restrict__ ipiv, int *__restrict__ info, int *queue)
{
    __shared__ int s_q;
    __shared__ FactorLds<T, W> sl;
    for (;;) {
        if (threadIdx.x == 0) s_q = atomicAdd(queue, 1);
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(s_q);  // uniform: bases in scalar registers
        __syncthreads();  // s_q is rewritten by the next ticket
        if (q >= batch) break;
        const int s = order[q];
        const SysDesc d = desc[s];
        Global<T> *a = (Global<T> *)A[s];
        Global<int> *piv = (Global<int> *)ipiv[s];
        // n < 0 marks a system whose sizes the allocation-free entry rejected
        int inf = d.n < 0 ? -1 : 0;
        if (d.n > 0) factor_system<T, W>(d.n, a, d.lda, piv, inf, sl);
        if (threadIdx.x == 0) info[s] = inf;
        __syncthreads();
    }
}

// The solves of every factored system (INFO = 0), by the same kind of
// persistent queue (queue[1]), after the factorization launch: a kernel of
// its own keeps its registers out of the factorization's.
template <typename T>
__global__ __launch_bounds__(FT) __attribute__((amdgpu_waves_per_eu(4))) void getrs_batched_kernel(
    int batch, const int *__restrict__ order, const SysDesc *__restrict__ desc,
    T *const *__restrict__ A, int *const *__restrict__ ipiv, T *const *__restrict__ B,
    const int *__restrict__ info, int *queue)
{
    __shared__ int s_q;
    __shared__ SolveLds<T> sl;
    for (;;) {
        if (threadIdx.x == 0) s_q = atomicAdd(queue + 1, 1);
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(s_q);
        __syncthreads();
        if (q >= batch) break;
        const int s = order[q];
        const SysDesc d = desc[s];
        if (d.n > 0 && d.nrhs > 0 && info[s] == 0)
            solve_all<T>(d.n, (const Global<T> *)A[s], d.lda, (const Global<int> *)ipiv[s],
                         (Global<T> *)B[s], d.ldb, d.nrhs, sl);
        __syncthreads();
    }
}

__global__ void zero_queue_kernel(int *q)
{
    if (threadIdx.x < 2 && blockIdx.x == 0) q[threadIdx.x] = 0;
}

// Set-up of the allocation-free entry, one workgroup: validates the device
// size arrays (a rejected system gets n = -1, i.e. INFO = -1, and no work),
// orders the systems largest n first by a counting sort (the order only
// balances the queue: every system's result is independent of it) and resets
// the queue.  Buckets: NMAX - n for a valid n, NMAX + 1 for a rejected one.
constexpr int PREP_BUCKETS = BATCHED_NMAX + 2;

__global__ __launch_bounds__(1024) void noalloc_prep_kernel(int batch, const int *__restrict__ n,
                                                            const int *__restrict__ nrhs,
                                                            const int *__restrict__ lda,
                                                            const int *__restrict__ ldb,
                                                            int *queue, int *order, SysDesc *desc)
{
    __shared__ int cnt[PREP_BUCKETS];
    for (int b = threadIdx.x; b < PREP_BUCKETS; b += blockDim.x) cnt[b] = 0;
    if (threadIdx.x < 2) queue[threadIdx.x] = 0;
    __syncthreads();
    for (int s = threadIdx.x; s < batch; s += blockDim.x) {
        const int ns = n[s], rs = nrhs[s], la = lda[s], lb = ldb[s];
        const bool ok = ns >= 0 && ns <= BATCHED_NMAX && rs >= 0 && rs <= BATCHED_NRHS_MAX &&
                        la >= max(1, ns) && lb >= max(1, ns);
        desc[s] = ok ? SysDesc{ns, rs, la, lb} : SysDesc{-1, 0, 1, 1};
        atomicAdd(&cnt[ok ? BATCHED_NMAX - ns : BATCHED_NMAX + 1], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {  // exclusive prefix sum of the bucket counts
        int run = 0;
        for (int b = 0; b < PREP_BUCKETS; b++) {
            const int c = cnt[b];
            cnt[b] = run;
            run += c;
        }
    }
    __syncthreads();
    for (int s = threadIdx.x; s < batch; s += blockDim.x) {
        const int ns = desc[s].n;  // written by this thread above
        order[atomicAdd(&cnt[ns >= 0 ? BATCHED_NMAX - ns : BATCHED_NMAX + 1], 1)] = s;
    }
}

// ---------------------------------------------------------------------------
// Synthetic systems for the tuner: A uniform[-1, 1) plus n I, B uniform.
__device__ __forceinline__ double hash_uniform(uint64_t x)
{
    x ^= x >> 33;
    x *= 0xff51afd7ed558ccdull;
    x ^= x >> 33;
    x *= 0xc4ceb9fe1a85ec53ull;
    x ^= x >> 33;
    return (double)(x >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}
template <typename T>
__global__ void fill_synthetic_kernel(int batch, const SysDesc *__restrict__ desc, T *const *A,
                                      T *const *B)
{
    for (int s = blockIdx.y; s < batch; s += gridDim.y) {
        const SysDesc d = desc[s];
        const size_t na = (size_t)d.lda * d.n, nbv = (size_t)d.ldb * d.nrhs;
        for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < na + nbv;
             e += (size_t)gridDim.x * 256) {
            const double u = hash_uniform(((uint64_t)s << 32) ^ e);
            if (e < na) {
                const int i = (int)(e % d.lda), j = (int)(e / d.lda);
                A[s][e] = (T)(u + (i == j ? (double)d.n : 0.0));
            } else {
                B[s][e - na] = (T)u;
            }
        }
    }
}

}  // namespace

// ============================================================================
// Host side
// ============================================================================
struct BatchedPlan {
    int batch = 0;
    std::vector<int> n, nrhs, lda, ldb;
    int *d_order = nullptr;
    SysDesc *d_desc = nullptr;
    int *d_queue = nullptr;
    void *graph_exec = nullptr;  // hipGraphExec_t of the last captured launch
    const void *g_key[4] = {nullptr, nullptr, nullptr, nullptr};
    int g_prec = -1, g_w = 0, g_wgs = 0;
    ~BatchedPlan()
    {
        if (graph_exec) (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph_exec));
        if (d_order) (void)hipFree(d_order);
        if (d_desc) (void)hipFree(d_desc);
        if (d_queue) (void)hipFree(d_queue);
    }
};

namespace {

bool same_sizes(const BatchedPlan &p, int batch, const int *n, const int *nrhs, const int *lda,
                const int *ldb)
{
    if (p.batch != batch) return false;
    for (int s = 0; s < batch; s++)
        if (p.n[s] != n[s] || p.nrhs[s] != nrhs[s] || p.lda[s] != lda[s] || p.ldb[s] != ldb[s])
            return false;
    return true;
}

template <typename T>
void launch(const BatchedPlan &p, int w, int wgs, int solve_wgs, T *const *A, int *const *ipiv,
            T *const *B, int *info, hipStream_t s)
{
    hipLaunchKernelGGL(zero_queue_kernel, dim3(1), dim3(64), 0, s, p.d_queue);
#define SLA_BATCHED(WV)                                                                          \
    hipLaunchKernelGGL((gesv_batched_kernel<T, WV>), dim3(wgs), dim3(FT), 0, s, p.batch,         \
                       p.d_order, p.d_desc, A, ipiv, info, p.d_queue)
    switch (w) {
    case 8: SLA_BATCHED(8); break;
    case 16: SLA_BATCHED(16); break;
    case 32: SLA_BATCHED(32); break;
    default: throw std::invalid_argument("batched: panel width must be 8, 16 or 32");
    }
#undef SLA_BATCHED
    SLA_LAUNCH_CHECK();
    hipLaunchKernelGGL(getrs_batched_kernel<T>, dim3(solve_wgs), dim3(FT), 0, s, p.batch,
                       p.d_order, p.d_desc, (T *const *)A, ipiv, B, info, p.d_queue);
    SLA_LAUNCH_CHECK();
}

}  // namespace

BatchedPlan &batched_plan(Handle &h, int batch, const int *n, const int *nrhs, const int *lda,
                          const int *ldb)
{
    if (!h.batched) h.batched = new BatchedPlan();
    BatchedPlan &p = *h.batched;
    if (same_sizes(p, batch, n, nrhs, lda, ldb)) return p;
    for (int s = 0; s < batch; s++) {
        if (n[s] < 0 || n[s] > BATCHED_NMAX || nrhs[s] < 0 || nrhs[s] > BATCHED_NRHS_MAX ||
            lda[s] < std::max(1, n[s]) || ldb[s] < std::max(1, n[s]))
            throw std::invalid_argument("batched: system " + std::to_string(s) +
                                        " has n, nrhs, lda or ldb out of range");
    }
    SLA_HIP(hipStreamSynchronize(h.stream));
    if (p.graph_exec) {
        SLA_HIP(hipGraphExecDestroy(static_cast<hipGraphExec_t>(p.graph_exec)));
        p.graph_exec = nullptr;
    }
    if (p.d_order) SLA_HIP(hipFree(p.d_order));
    if (p.d_desc) SLA_HIP(hipFree(p.d_desc));
    if (!p.d_queue) SLA_HIP(hipMalloc(&p.d_queue, 64));
    p.batch = batch;
    p.n.assign(n, n + batch);
    p.nrhs.assign(nrhs, nrhs + batch);
    p.lda.assign(lda, lda + batch);
    p.ldb.assign(ldb, ldb + batch);
    // largest work first (n^3 + n^2 nrhs), ties by index
    std::vector<int> order(batch);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        const double wx = (double)n[x] * n[x] * (n[x] + 3.0 * nrhs[x]);
        const double wy = (double)n[y] * n[y] * (n[y] + 3.0 * nrhs[y]);
        return wx > wy;
    });
    std::vector<SysDesc> desc(batch);
    for (int s = 0; s < batch; s++) desc[s] = SysDesc{n[s], nrhs[s], lda[s], ldb[s]};
    SLA_HIP(hipMalloc(&p.d_order, sizeof(int) * std::max(1, batch)));
    SLA_HIP(hipMalloc(&p.d_desc, sizeof(SysDesc) * std::max(1, batch)));
    SLA_HIP(hipMemcpy(p.d_order, order.data(), sizeof(int) * batch, hipMemcpyHostToDevice));
    SLA_HIP(hipMemcpy(p.d_desc, desc.data(), sizeof(SysDesc) * batch, hipMemcpyHostToDevice));
    return p;
}

void batched_plan_free(BatchedPlan *p) { delete p; }

}  // namespace sla

// ---------------------------------------------------------------------------
// Allocation-free entry: the queue counter, the order and the size
// descriptors live in this fixed device array (one copy per GPU, kept until
// the process ends) instead of memory the library allocates.  Layout: queue
// at 0, order at 256, descriptors after BATCHED_NOALLOC_MAX ints.
static __device__ __align__(256) unsigned char
    scratch[256 + (size_t)sla::BATCHED_NOALLOC_MAX * (sizeof(int) + 4 * sizeof(int))];

namespace sla {

namespace {

std::mutex g_scratch_mu;
void *g_scratch_ptr[64] = {};  // device address of `scratch` on each GPU

// Device address of this GPU's `scratch` (looked up once per device, with
// that device current; host code never uses the array's name as an address).
void *noalloc_scratch(int device)
{
    if (device < 0 || device >= 64) throw std::runtime_error("batched: device id out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        SLA_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) throw std::runtime_error("batched: no device address for the scratch array");
        g_scratch_ptr[device] = p;
    }
    return g_scratch_ptr[device];
}

}  // namespace

template <typename T>
void gesv_batched_noalloc_device(Handle &h, int batch, const int *dn, const int *dnrhs,
                                 T *const *dA, const int *dlda, int *const *dipiv, T *const *dB,
                                 const int *dldb, int *dinfo)
{
    if (batch < 0 || batch > BATCHED_NOALLOC_MAX)
        throw std::invalid_argument("batched (no allocation): batch above " +
                                    std::to_string(BATCHED_NOALLOC_MAX) + " systems");
    int cur = -1;
    SLA_HIP(hipGetDevice(&cur));
    if (cur != h.device)
        throw std::runtime_error("batched (no allocation): the handle's device must be current");
    if (batch == 0) return;
    static_assert(sizeof(SysDesc) == 4 * sizeof(int), "descriptor layout of the scratch array");
    char *base = static_cast<char *>(noalloc_scratch(cur));
    int *queue = reinterpret_cast<int *>(base);
    int *order = reinterpret_cast<int *>(base + 256);
    SysDesc *desc = reinterpret_cast<SysDesc *>(base + 256 + sizeof(int) * BATCHED_NOALLOC_MAX);
    hipLaunchKernelGGL(noalloc_prep_kernel, dim3(1), dim3(1024), 0, h.stream, batch, dn, dnrhs,
                       dlda, dldb, queue, order, desc);
    SLA_LAUNCH_CHECK();
    const int wgs = std::max(1, h.batched_wgs_per_cu) * h.num_cus;
#define SLA_BATCHED(WV)                                                                          \
    hipLaunchKernelGGL((gesv_batched_kernel<T, WV>), dim3(wgs), dim3(FT), 0, h.stream, batch,     \
                       order, desc, dA, dipiv, dinfo, queue)
    switch (h.batched_w) {
    case 8: SLA_BATCHED(8); break;
    case 16: SLA_BATCHED(16); break;
    case 32: SLA_BATCHED(32); break;
    default: throw std::invalid_argument("batched: panel width must be 8, 16 or 32");
    }
#undef SLA_BATCHED
    SLA_LAUNCH_CHECK();
    hipLaunchKernelGGL(getrs_batched_kernel<T>, dim3(SOLVE_WGS * h.num_cus), dim3(FT), 0, h.stream, batch,
                       order, desc, (T *const *)dA, (int *const *)dipiv, dB, dinfo, queue);
    SLA_LAUNCH_CHECK();
}

template void gesv_batched_noalloc_device<double>(Handle &, int, const int *, const int *,
                                                  double *const *, const int *, int *const *,
                                                  double *const *, const int *, int *);
template void gesv_batched_noalloc_device<float>(Handle &, int, const int *, const int *,
                                                 float *const *, const int *, int *const *,
                                                 float *const *, const int *, int *);

template <typename T>
void gesv_batched_device(Handle &h, int batch, const int *n, const int *nrhs, T *const *dA,
                         const int *lda, int *const *dipiv, T *const *dB, const int *ldb, int *dinfo)
{
    if (batch <= 0) return;
    BatchedPlan &p = batched_plan(h, batch, n, nrhs, lda, ldb);
    const int w = h.batched_w;
    const int wgs = std::max(1, h.batched_wgs_per_cu) * h.num_cus;
    const int prec = sizeof(T) == 8 ? 0 : 1;
    if (!h.batched_graph) {
        launch<T>(p, w, wgs, SOLVE_WGS * h.num_cus, dA, dipiv, dB, dinfo, h.stream);
        SLA_HIP(hipStreamSynchronize(h.stream));
        return;
    }
    // hipGraph path: the queue reset (a kernel, not a memset) and the
    // persistent launch captured once per (pointer arrays, sizes, shape)
    // and replayed afterwards.
    const void *key[4] = {dA, dipiv, dB, dinfo};
    const bool hit = p.graph_exec && std::equal(key, key + 4, p.g_key) && p.g_prec == prec &&
                     p.g_w == w && p.g_wgs == wgs;
    if (!hit) {
        if (p.graph_exec) {
            SLA_HIP(hipGraphExecDestroy(static_cast<hipGraphExec_t>(p.graph_exec)));
            p.graph_exec = nullptr;
        }
        hipStream_t cs = h.own_stream;  // capture on the handle's own stream
        SLA_HIP(hipStreamSynchronize(h.stream));
        hipGraph_t g = nullptr;
        SLA_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        try {
            launch<T>(p, w, wgs, SOLVE_WGS * h.num_cus, dA, dipiv, dB, dinfo, cs);
        } catch (...) {
            (void)hipStreamEndCapture(cs, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        SLA_HIP(hipStreamEndCapture(cs, &g));
        hipGraphExec_t ge = nullptr;
        SLA_HIP(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
        SLA_HIP(hipGraphDestroy(g));
        p.graph_exec = ge;
        std::copy(key, key + 4, p.g_key);
        p.g_prec = prec;
        p.g_w = w;
        p.g_wgs = wgs;
    }
    SLA_HIP(hipGraphLaunch(static_cast<hipGraphExec_t>(p.graph_exec), h.stream));
    SLA_HIP(hipStreamSynchronize(h.stream));
}

template void gesv_batched_device<double>(Handle &, int, const int *, const int *, double *const *,
                                          const int *, int *const *, double *const *, const int *,
                                          int *);
template void gesv_batched_device<float>(Handle &, int, const int *, const int *, float *const *,
                                         const int *, int *const *, float *const *, const int *,
                                         int *);

// Autotuner: times every (panel width, workgroups per CU) on synthetic
// systems of the given sizes (diagonally dominant, so every candidate does
// the same work) and keeps the fastest in the handle.
template <typename T>
BatchedTune tune_batched_device(Handle &h, int batch, const int *n, const int *nrhs, int reps)
{
    BatchedTune out;
    if (batch <= 0) return out;
    std::vector<int> lda(batch), ldb(batch);
    size_t total = 0, total_piv = 0;
    for (int s = 0; s < batch; s++) {
        lda[s] = std::max(1, n[s]);
        ldb[s] = std::max(1, n[s]);
        total += (size_t)lda[s] * n[s] + (size_t)ldb[s] * nrhs[s];
        total_piv += (size_t)std::max(1, n[s]);
    }
    BatchedPlan &p = batched_plan(h, batch, n, nrhs, lda.data(), ldb.data());
    T *data = nullptr;
    int *piv = nullptr, *info = nullptr;
    void **ptrs = nullptr;
    SLA_HIP(hipMalloc(&data, total * sizeof(T) + 256));
    SLA_HIP(hipMalloc(&piv, total_piv * sizeof(int) + 256));
    SLA_HIP(hipMalloc(&info, sizeof(int) * batch));
    SLA_HIP(hipMalloc(&ptrs, sizeof(void *) * 3 * batch));
    std::vector<void *> hp(3 * (size_t)batch);
    size_t off = 0, offp = 0;
    for (int s = 0; s < batch; s++) {
        hp[s] = data + off;
        off += (size_t)lda[s] * n[s];
        hp[2 * (size_t)batch + s] = data + off;
        off += (size_t)ldb[s] * nrhs[s];
        hp[(size_t)batch + s] = piv + offp;
        offp += (size_t)std::max(1, n[s]);
    }
    SLA_HIP(hipMemcpy(ptrs, hp.data(), sizeof(void *) * hp.size(), hipMemcpyHostToDevice));
    T *const *dA = reinterpret_cast<T *const *>(ptrs);
    int *const *dP = reinterpret_cast<int *const *>(ptrs + batch);
    T *const *dB = reinterpret_cast<T *const *>(ptrs + 2 * (size_t)batch);
    hipEvent_t e0, e1;
    SLA_HIP(hipEventCreate(&e0));
    SLA_HIP(hipEventCreate(&e1));
    double best = 1e30;
    for (int w : {8, 16, 32})
        for (int k : {1, 2, 4}) {
            double ms_sum = 0.0;
            for (int r = 0; r < reps + 1; r++) {
                hipLaunchKernelGGL(fill_synthetic_kernel<T>, dim3(64, std::min(batch, 65535)), dim3(256), 0, h.stream,
                                   batch, p.d_desc, dA, dB);
                SLA_HIP(hipEventRecord(e0, h.stream));
                launch<T>(p, w, k * h.num_cus, SOLVE_WGS * h.num_cus, dA, dP, dB, info, h.stream);
                SLA_HIP(hipEventRecord(e1, h.stream));
                SLA_HIP(hipEventSynchronize(e1));
                float ms = 0.f;
                SLA_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (r > 0) ms_sum += ms;  // the first run warms up
            }
            const double ms = ms_sum / std::max(1, reps);
            out.tried.push_back({w, k, ms});
            if (ms < best) {
                best = ms;
                out.w = w;
                out.wgs_per_cu = k;
                out.ms = ms;
            }
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(data);
    (void)hipFree(piv);
    (void)hipFree(info);
    (void)hipFree(ptrs);
    h.batched_w = out.w;
    h.batched_wgs_per_cu = out.wgs_per_cu;
    return out;
}

template BatchedTune tune_batched_device<double>(Handle &, int, const int *, const int *, int);
template BatchedTune tune_batched_device<float>(Handle &, int, const int *, const int *, int);

}  // namespace sla
