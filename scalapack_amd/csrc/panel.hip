// panel.hip -- the unblocked panel factorization PDGETF2 (SRC/pdgetf2.f:206-237)
// for a tall leaf of at most W columns, as one launch of G resident
// workgroups that hold the leaf in registers.
//
// Per column j the reference does PDAMAX (pivot search) -> PDSWAP (row
// interchange) -> PDSCAL(1/GMAX) -> PDGER(-1) (rank-1 update).  Here no row
// changes place while the leaf is factored: every row carries the position
// the interchanges have brought it to, a row whose position is below j is
// done, and the interchange of j and p is an exchange of two positions.
//   1. every wave finds the largest |v| among its rows of position >= j (ties
//      to the lowest position, as IDAMAX) and posts that row to LDS together
//      with 1 / v; one workgroup barrier; every wave folds the posts itself;
//   2. with more than one workgroup, each publishes its candidate (value,
//      position and row) in mailbox words of column j; each word is written
//      once per launch and starts out empty, so a word that is no longer empty
//      holds this column's value: no counter, no barrier.  Every wave gathers
//      the G values and positions, reduces them in the same total order, so
//      all agree on p, and fetches that row;
//   3. rows of position > j are scaled by the reciprocal (the reference's
//      ONE / GMAX multiply, pdgetf2.f:224) and updated a -= l * u with one fma.
// The rows are written to their final positions at the end, and PDGETF2's
// interchanges of the other columns of the block column (pdgetf2.f:219-220)
// follow as the leaf's net row permutation (no other access touches those
// columns meanwhile, so the result is the same as swapping per column).
// A zero pivot skips the interchange and the scaling and records the first
// such column (pdgetf2.f:226-228); the update still runs, as PDGER does.
//
// What bounds it is the latency of that chain, W times per leaf.  Two choices
// shorten it.  A row lies in the four lanes of a quad, column c in lane c % 4
// (register c / 4): the pivot row costs a lane NC LDS reads instead of W, the
// posting quad writes it with NC / 2 16-byte stores, and the multiplier reaches
// the quad by one DPP move.  And the column loop is a run-time loop whose body
// handles one column and rotates the registers by one after every fourth, so
// that every register index is a constant in a body of a few KB: unrolled over
// all columns, as before, the leaf was 340 KB of code that every launch fetched
// anew.
//
// The exchange is as fast as the path between the workgroups: a word written
// and read through the L2 of one XCD takes 230 ns, through the device-coherent
// path 440 ns within an XCD and 500 - 620 ns between two (ping-pong of two
// workgroups).  So a leaf of at most 32 workgroups puts them all on one XCD, a
// different one from leaf to leaf, because the trailing update beside it is
// dealt evenly over all of them.  Where that takes more than a quarter of the XCD,
// leaves of several handles could keep each other from getting all their
// workgroups to run; there the leaf gives way after 200 us in column 0 and a second
// launch, over all XCDs, does the work (sla_panel_plan.h).  That launch costs a
// leaf that did not give way 6 us.  The pivot row is fetched once the pivot is
// known: gathering all G candidate rows in one trip, to LDS, took 85 us at m =
// 2000 where this takes 77, and 57 KB of LDS where this takes 13.
//
// A workgroup of four waves with at most 128 registers starts beside the
// trailing update (which leaves that much of every CU free, gemm_tile.hip).
// There it takes 180 - 220 us instead of 80: every instruction of its chain
// waits for the update's.
//
// Measured on 32 FP64 columns, alone on the GPU, us per leaf, before (all
// columns unrolled, rows interchanged in registers, the workgroups spread over
// the XCDs) and now: m = 100: 120, 36; 1000: 130, 73; 4096: 149, 79; 8192: 157,
// 82; 16384: 165, 108; 32768: 182, 132.
//
// Mailbox: two regions of 32 column blocks; launch L uses region L & 1 and
// refills the words launch L - 1 wrote in region (L + 1) & 1 -- that launch
// has finished -- with the empty pattern, so that launch L + 1 finds its
// region empty.
#include "sla_common.h"
#include "sla_kernels.h"
#include "sla_panel_plan.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace sla {

namespace {

constexpr int NWV = 8;           // waves per workgroup at most
static_assert(LEAF_GMAX <= PANEL_MAIL_GMAX, "mailbox too small for the leaf's grid");

constexpr uint64_t MAIL_EMPTY = ~0ull;  // no position or value word has this pattern

// Storage of one value in a mailbox word.  A double whose bits equal the
// empty pattern (a NaN) is stored as the neighbouring NaN pattern.
__device__ __forceinline__ uint64_t mail_word(double x)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    return b == MAIL_EMPTY ? MAIL_EMPTY - 1 : b;
}
__device__ __forceinline__ uint64_t mail_word(float x)
{
    return (uint64_t)__builtin_bit_cast(uint32_t, x);
}
template <typename T>
__device__ __forceinline__ T mail_value(uint64_t w)
{
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, w);
    else return __builtin_bit_cast(T, (uint32_t)w);
}

// Pivot key of a candidate: monotone in |v|, more than 1 for a nonzero v; 0
// for no candidate and for a NaN, which IDAMAX's comparisons never select.  A
// NaN in row j itself (top) counts as a zero: a column without anything larger
// keeps row j.
__device__ __forceinline__ uint64_t mag_key(double v, bool valid, bool top)
{
    const double a = fabs(v);
    return !valid ? 0ull : a == a ? __builtin_bit_cast(uint64_t, a) + 1ull : (top ? 1ull : 0ull);
}
__device__ __forceinline__ uint64_t mag_key(float v, bool valid, bool top)
{
    return mag_key((double)v, valid, top);
}

// The wave's first maximum by full keys: the lane holding the largest key and,
// among equal keys, the lowest position; its key and position in every lane.
__device__ __forceinline__ int wave_pick(uint64_t &key, int &pos)
{
    const uint32_t hi = (uint32_t)(key >> 32), lo = (uint32_t)key;
    const uint32_t hm = wave_max(hi);
    const uint32_t lm = wave_max(hi == hm ? lo : 0u);
    const bool in = hi == hm && lo == lm;
    const uint32_t np = in ? ~(uint32_t)pos : 0u;  // positions are >= 0
    const uint32_t nm = wave_max(np);
    const int l = __builtin_ctzll(__ballot(in && np == nm));
    const uint32_t kl = __builtin_amdgcn_readlane(lo, l), kh = __builtin_amdgcn_readlane(hi, l);
    key = ((uint64_t)kh << 32) | kl;
    pos = __builtin_amdgcn_readlane(pos, l);
    return l;
}

// The leading 32 bits of |v|, monotone in |v|.  One maximum of them decides a
// pivot search unless it is shared (the rest of the bits, then the position
// decide), is zero (zeros, denormals, no row) or is not finite; those searches
// use the full keys.
__device__ __forceinline__ uint32_t mag_hi(double v)
{
    return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32) & 0x7fffffffu;
}
__device__ __forceinline__ uint32_t mag_hi(float v)
{
    return __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
}
template <typename T>
__device__ __forceinline__ bool decides(uint32_t hm)
{
    return hm - 1u < (sizeof(T) == 8 ? 0x7ff00000u : 0x7f800000u) - 1u;
}

// v[q] <- the value of lane S of the quad, in all four lanes.
template <int S, int NQ>
__device__ __forceinline__ void quad_bcast(double (&v)[NQ])
{
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v[q]);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, S * 0x55, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), S * 0x55, 0xf, 0xf, false);
        v[q] = __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
    }
}
template <int S, int NQ>
__device__ __forceinline__ void quad_bcast(float (&v)[NQ])
{
#pragma unroll
    for (int q = 0; q < NQ; q++)
        v[q] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                             0, __builtin_bit_cast(int, v[q]), S * 0x55, 0xf, 0xf, false));
}

// A row in LDS: 4 NC values in register order, lane by lane; 34 words apart, which
// spreads one column of all rows over the banks and keeps them 16-byte aligned.
constexpr int CWL = 34;

template <typename T>
struct alignas(16) LeafLds {
    T wrow[2][NWV][CWL];          // each wave's candidate, by column parity
    int wpos[2][NWV];             // its position; INT_MAX: no candidate
    T prow[NWV][CWL];             // the pivot row, a copy for each wave that fetched it
    T u[32][CWL];                 // the pivot rows of the leaf
    int s_pv[32];                 // interchange of each column; -1: a zero pivot, none
    int s_dst[64], s_src[64], s_npair;
    int s_abort[2];               // a wait gave up, by column parity
};

struct LeafArgs {
    uint64_t *box;  // this launch's mailbox region
    int *abort_flag;
    uint64_t spin_limit, t0;
    // of a leaf that may give way:
    unsigned *yield;    // where it says so (null: it does not)
    unsigned yield_id;  // by this number
    uint64_t patience;  // ticks it waits in column 0 before it does
    int G, g;       // workgroups of the leaf, this one
    uint32_t xcd;   // the die it runs on
};

// A word for the other workgroups: through the L2 of the XCD (local: every
// workgroup of the leaf runs on this one, and a load that bypasses the L1 finds
// it there) or to where every XCD sees it.  The local store has workgroup scope,
// which promises other workgroups nothing in the language: that they see it rests on
// the one L2 of an XCD, to which the L1 writes every store through.  A word that did
// not arrive would end in the bounded wait's error, not in a wrong pivot.
__device__ __forceinline__ void post_word(uint64_t *p, uint64_t v, bool local)
{
    if (local) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else coherent_store(p, v);
}

// Publishes the workgroup's candidate of column j: its row, its value and its
// position (INT_MAX: none), whose word's upper half carries the XCD.  One wave.
template <typename T, int NC>
__device__ __forceinline__ void publish(const LeafArgs &ar, uint64_t *cb, bool local, const T *src,
                                        T val, int cpos, int lane)
{
    constexpr int NV = 4 * NC;  // values of a row
    if (lane < NV + 2) {
        const int at = lane < NV ? ar.g * PANEL_MAIL_CW + lane
                                 : (lane == NV ? PANEL_MAIL_VAL : PANEL_MAIL_POS) + ar.g;
        const uint64_t w = lane < NV   ? mail_word(src[lane])
                         : lane == NV ? mail_word(val)
                                      : ((uint64_t)ar.xcd << 32) | (uint32_t)cpos;
        post_word(&cb[at], w, local);
    }
}

// Whether a wait of column j goes on: false after spin_limit, when another wait gave
// up, or when the leaf gives way.  A leaf gives way only in column 0: a workgroup
// that leaves there posts nothing more, so no other one gets past column 1, and
// since nothing but the mailbox is written before the last column, all leave the
// matrix as it was.  Once column 0 is through, every workgroup runs.
template <bool YIELDS>
__device__ __forceinline__ bool keep_waiting(const LeafArgs &ar, int j, unsigned &it, int *s_abort)
{
    // without patience it looks at once
    if ((++it & 15u) != 0 && !(YIELDS && ar.yield && ar.patience == 0)) return true;
    bool on = true;
    const uint64_t dt = wall_clock64() - ar.t0;
    if (coherent_load(ar.abort_flag)) on = false;
    else if (YIELDS && ar.yield && coherent_load(ar.yield) == ar.yield_id) on = false;
    else if (YIELDS && ar.yield && j == 0 && dt > ar.patience) {
        coherent_store(ar.yield, ar.yield_id);
        on = false;
    } else if (dt > ar.spin_limit) {
        coherent_store(ar.abort_flag, 1);
        on = false;
    }
    if (!on) *s_abort = 1;
    return on;
}

// x[0] .. x[NC-1] rotated down by one.  Written out by recursion: as a loop it
// may become a memmove, which keeps the array in scratch memory.
template <int NC, int I = 0, typename T>
__device__ __forceinline__ void rotate_row(T (&x)[NC], T first)
{
    if constexpr (I + 1 < NC) {
        x[I] = x[I + 1];
        rotate_row<NC, I + 1>(x, first);
    } else {
        x[I] = first;
    }
}

// x[q][i] -= l[q] u[i] for 1 <= i < live (uniform).
template <int I = 1, int NQ, int NC, typename T>
__device__ __forceinline__ void update_rows(T (&x)[NQ][NC], const T (&l)[NQ], const T (&u)[NC],
                                            int live)
{
    if constexpr (I < NC) {
        if (I < live) {
#pragma unroll
            for (int q = 0; q < NQ; q++) x[q][I] = fma(-l[q], u[I], x[q][I]);
            update_rows<I + 1>(x, l, u, live);
        }
    }
}

// Column j, in register 0 of the lanes with cg = j % 4 = S; the registers
// 1 .. live-1 hold the columns further right.  A row that is done (or beyond
// the leaf) holds zeros there, so it neither wins a search nor is changed by an
// update; its multipliers stay.
template <typename T, int NC, int NQ, bool SOLO, bool YIELDS>
__device__ __forceinline__ void leaf_step(const LeafArgs &ar, int j, T (&a)[NQ][NC],
                                          int (&pos)[NQ], bool &local, bool &dead, LeafLds<T> &sl)
{
    typedef T v2_t __attribute__((ext_vector_type(2)));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, cg = lane & 3;
    const int nw = (int)blockDim.x >> 6, pb = j & 1, S = j & 3, live = NC - (j >> 2);

    // 1. candidate of the wave: row q of lane wl
    int wl = 0, uq = 0;
    bool found;
    {
        const uint64_t cols = 0x1111111111111111ull << S;  // the lanes holding column j
        uint32_t h[NQ], hx = 0;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            h[q] = mag_hi(a[q][0]);
            hx = h[q] > hx ? h[q] : hx;
        }
        const uint32_t hm = wave_max(cg == S ? hx : 0u);
        int cnt = 0;
        uint64_t t = 0;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const uint64_t tq = __ballot(h[q] == hm) & cols;
            cnt += __builtin_popcountll(tq);
            uq = tq ? q : uq;
            t |= tq;
        }
        found = true;
        if (cnt == 1 && decides<T>(hm)) {
            wl = __builtin_ctzll(t);
        } else {
            uint64_t bk = 0;
            int bp = INT_MAX, bq = 0;
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                const uint64_t k = mag_key(a[q][0], cg == S && pos[q] >= j, pos[q] == j);
                const bool take = k > bk || (k != 0 && k == bk && pos[q] < bp);
                bk = take ? k : bk;
                bp = take ? pos[q] : bp;
                bq = take ? q : bq;
            }
            wl = wave_pick(bk, bp);
            uq = __builtin_amdgcn_readlane(bq, wl);
            found = bk != 0;
        }
    }
    if (found && (lane >> 2) == (wl >> 2)) {
        T *dst = &sl.wrow[pb][wave][cg * NC];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            if (uq == q) {
#pragma unroll
                for (int i = 0; i < NC; i += 2) {
                    const v2_t x = {a[q][i], a[q][i + 1]};
                    *reinterpret_cast<v2_t *>(&dst[i]) = x;
                }
                sl.wpos[pb][wave] = pos[q];
                // keeps the branches apart: merged, they select a row by
                // address, and the array goes to scratch memory
                asm volatile("; row %0" ::"i"(q));
            }
        }
    }
    if (!found && lane == 0) sl.wpos[pb][wave] = INT_MAX;
    __syncthreads();
    // a wait of the column before that gave up: all waves see it here, and the
    // workgroup posts nothing of this column
    if (!SOLO) dead = sl.s_abort[pb ^ 1] != 0;
    // the workgroup's: lane x looks at the candidate of wave x % 8
    int p, fw;
    bool nonzero = true;
    T pv;
    {
        const int x = lane & (NWV - 1);
        const int xp = x < nw ? sl.wpos[pb][x] : INT_MAX;
        const T xv = sl.wrow[pb][x][S * NC];
        const uint32_t h = xp != INT_MAX ? mag_hi(xv) : 0u;
        uint32_t hm = dpp_max<0x121, 0xf>(h);
        hm = dpp_max<0x122, 0xf>(hm);
        hm = dpp_max<0x124, 0xf>(hm);
        hm = (uint32_t)__builtin_amdgcn_readfirstlane((int)hm);
        const unsigned t = (unsigned)__ballot(h == hm) & ((1u << NWV) - 1u);
        if (decides<T>(hm) && (t & (t - 1)) == 0) {
            fw = __builtin_ctz(t);
            p = __builtin_amdgcn_readlane(xp, fw);
        } else {
            uint64_t ck = mag_key(xv, xp != INT_MAX, xp == j);
            p = ck != 0 ? xp : INT_MAX;
            fw = wave_pick(ck, p) & (NWV - 1);
            nonzero = ck > 1;
        }
        pv = lane_read(xv, fw);
    }
    const T *prow = sl.wrow[pb][fw];
    T u[NC];

    // 2. the other workgroups
    if constexpr (!SOLO) {
        uint64_t *cb = ar.box + (size_t)j * PANEL_MAIL_COL;
        if (wave == nw - 1 && !dead) publish<T, NC>(ar, cb, local, prow, pv, p, lane);
        const int G = ar.G;
        // values and positions of candidates lane and lane + 64
        uint64_t kv[2], kp[2];
        unsigned it = 0;
        const int x0 = min(lane, G - 1), x1 = min(lane + 64, G - 1);
        do {
            kv[0] = coherent_load(&cb[PANEL_MAIL_VAL + x0]);
            kp[0] = coherent_load(&cb[PANEL_MAIL_POS + x0]);
            kv[1] = kv[0];
            kp[1] = kp[0];
            if (G > 64) {
                kv[1] = coherent_load(&cb[PANEL_MAIL_VAL + x1]);
                kp[1] = coherent_load(&cb[PANEL_MAIL_POS + x1]);
            }
        } while ((kv[0] == MAIL_EMPTY || kp[0] == MAIL_EMPTY || kv[1] == MAIL_EMPTY ||
                  kp[1] == MAIL_EMPTY) &&
                 keep_waiting<YIELDS>(ar, j, it, &sl.s_abort[pb]));
        int xp = lane < G ? (int)kp[0] : INT_MAX;
        T xv = mail_value<T>(kv[0]);
        const uint32_t h = xp != INT_MAX ? mag_hi(xv) : 0u;
        const uint32_t hm = wave_max(h);
        const uint64_t t = __ballot(h == hm);
        nonzero = true;
        int gw;
        if (G <= 64 && decides<T>(hm) && (t & (t - 1)) == 0) {
            gw = __builtin_ctzll(t);
            p = __builtin_amdgcn_readlane(xp, gw);
            pv = lane_read(xv, gw);
        } else {
            uint64_t ck = mag_key(xv, xp != INT_MAX, xp == j);
            int bg = lane;
            if (G > 64) {
                const int yp = lane + 64 < G ? (int)kp[1] : INT_MAX;
                const T yv = mail_value<T>(kv[1]);
                const uint64_t yk = mag_key(yv, yp != INT_MAX, yp == j);
                if (yk > ck || (yk == ck && yp < xp)) {
                    ck = yk;
                    xp = yp;
                    xv = yv;
                    bg = lane + 64;
                }
            }
            p = ck != 0 ? xp : INT_MAX;
            const int l = wave_pick(ck, p);
            gw = __builtin_amdgcn_readlane(bg, l);
            nonzero = ck > 1;
            pv = lane_read(xv, l);
        }
        if (j == 0) {
            // from here on through the L2, if every workgroup is on this XCD
            local = __all((kp[0] >> 32) == ar.xcd && (kp[1] >> 32) == ar.xcd);
        }
        // the pivot row: a word a lane (one request for the 256 bytes), then
        // through the wave's own slot in LDS
        const uint64_t *rw = cb + (size_t)gw * PANEL_MAIL_CW + lane % (4 * NC);
        uint64_t w;
        while ((w = coherent_load(rw)) == MAIL_EMPTY && keep_waiting<YIELDS>(ar, j, it, &sl.s_abort[pb])) {
        }
        if (lane < 4 * NC) sl.prow[wave][lane] = mail_value<T>(w);
        prow = sl.prow[wave];
    }
#pragma unroll
    for (int i = 0; i < NC; i += 2) {
        const v2_t x = *reinterpret_cast<const v2_t *>(&prow[cg * NC + i]);
        u[i] = x[0];
        u[i + 1] = x[1];
    }
    if (wave == (j & (nw - 1)) && lane < 4 * NC) sl.u[j][lane] = prow[lane];

    // 3. interchange, scaling, rank-1 update
    T l[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) l[q] = a[q][0];
    if (S == 0) quad_bcast<0>(l);
    else if (S == 1) quad_bcast<1>(l);
    else if (S == 2) quad_bcast<2>(l);
    else quad_bcast<3>(l);
    // a zero pivot keeps row j (p = j) and leaves the column unscaled
    const T rcp = nonzero ? T(1) / pv : T(1);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int x = pos[q];
        const bool own = x == p;
        pos[q] = own ? j : (x == j ? p : x);
        // the pivot row with l = 1 becomes zero right of the diagonal
        l[q] = own ? T(1) : l[q] * rcp;
    }
    if (tid == 0) sl.s_pv[j] = nonzero ? p : -1;
    if (cg >= S) {
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const T x0 = fma(-l[q], u[0], a[q][0]);
            a[q][0] = cg == S ? l[q] : x0;
        }
    }
    update_rows(a, l, u, live);
}

// NC: registers per row and lane (leaf width 4 NC), NQ: rows per quad; a wave
// holds 16 NQ rows.  SOLO: a single workgroup, no exchange.
// stride: the leaf's workgroups are every stride-th of the launch (the others
// leave at once): with 8, the number of XCDs over which consecutive workgroups
// are dealt, they share one XCD and its L2 (checked in column 0).
// yield_id: number by which the leaf gives way in *yield (0: it does not);
// after_id: the leaf runs only if the launch of that number did (0: always).
// YIELDS: the leaf may give way, or runs after one that may have; the others go
// without that code, which costs them scalar registers and 1 to 3 us.
// Scratch, FP64: five or six values a lane of the 32-column leaves at WPE = 4, stored
// before the column loop and read after it; 68 and 92 bytes of the 8-column leaves with
// 64 values a lane, within it.
template <typename T, int NC, int NQ, bool SOLO, int PT, int WPE, bool YIELDS>
__global__ __launch_bounds__(PT) __attribute__((amdgpu_waves_per_eu(WPE))) void panel_leaf_kernel(
    T *__restrict__ A, int lda, int m, int wa, int lcols, int rcols, int row0, int col0,
    int *__restrict__ ipiv, uint64_t *__restrict__ mail, int region, int prev_wa, int prev_g,
    int *abort_flag, int *zero_col, uint64_t spin_limit, int stride, int first, unsigned *yield,
    unsigned yield_id, unsigned after_id, uint64_t patience)
{
    if (!SOLO && (int)blockIdx.x % stride != first) return;
    const int G = SOLO ? 1 : gridDim.x / stride, g = SOLO ? 0 : blockIdx.x / stride;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, nw = (int)blockDim.x >> 6;
    const int cg = lane & 3, rg = lane >> 2;
    const int base = (g * nw + wave) * (16 * NQ) + rg;  // row q of this quad: base + 16 q

    __shared__ LeafLds<T> sl;
    if (tid < 2) sl.s_abort[tid] = 0;

    if constexpr (!SOLO) {
        // empty the words the previous launch that used the mailbox wrote (the
        // other region): columns < prev_wa, its prev_g candidates
        uint64_t *o = mail + (size_t)(region ^ 1) * PANEL_MAIL_REGION;
        const int per = prev_g * (PANEL_MAIL_CW + 2);
        for (int jj = 0; jj < prev_wa; jj++)
            for (int e = g * (int)blockDim.x + tid; e < per; e += G * (int)blockDim.x)
                coherent_store(&o[(size_t)jj * PANEL_MAIL_COL +
                                  (e < prev_g * PANEL_MAIL_CW ? e
                                   : e < prev_g * (PANEL_MAIL_CW + 1)
                                       ? PANEL_MAIL_VAL + e - prev_g * PANEL_MAIL_CW
                                       : PANEL_MAIL_POS + e - prev_g * (PANEL_MAIL_CW + 1))],
                               MAIL_EMPTY);
        if (YIELDS && after_id != 0 && coherent_load(yield) != after_id) return;
    }

    // column 4 i + cg of the leaf in register i; columns right of a narrow
    // leaf are zeros that no step pivots on
    T a[NQ][NC];
    int pos[NQ];  // current position of the row; -1: no row
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int r = base + 16 * q;
        pos[q] = r < m ? r : -1;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int c = 4 * i + cg;
            a[q][i] = (r < m && c < wa) ? A[r + (size_t)c * lda] : T(0);
        }
    }
    const LeafArgs ar{mail + (size_t)region * PANEL_MAIL_REGION, abort_flag, spin_limit, (uint64_t)wall_clock64(),
                      YIELDS && yield_id != 0 ? yield : nullptr, yield_id, patience, G, g,
                      SOLO ? 0u : (uint32_t)__builtin_amdgcn_s_getreg(63508) & 0xffffu};  // XCC_ID
    bool local = false;
    __syncthreads();
    // After the last column of a group of four the registers rotate by one.
    // Nothing in the loop writes to global memory but the exchange: the waits
    // for a store's completion would join the chain.
    bool dead = false;  // uniform
#pragma unroll 1
    for (int t = 0; t < NC && !dead; t++) {
#pragma unroll 1
        for (int j = 4 * t; j < min(4 * t + 4, wa) && !dead; j++)
            leaf_step<T, NC, NQ, SOLO, YIELDS>(ar, j, a, pos, local, dead, sl);
#pragma unroll
        for (int q = 0; q < NQ; q++) rotate_row<NC>(a[q], a[q][0]);
    }

    // Every row to its final position (every workgroup has loaded its rows:
    // it took part in the last column's exchange).  NC rotations have brought
    // every column back to its register.  Of a pivot row the multipliers are
    // here; its part of U is in sl.u, in the register order of its column.
    __syncthreads();
    if (!SOLO && (sl.s_abort[0] | sl.s_abort[1])) return;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        if (pos[q] >= 0) {
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const int c = 4 * i + cg;
                if (c < wa && (pos[q] >= wa || c < pos[q])) A[pos[q] + (size_t)c * lda] = a[q][i];
            }
        }
    }
    if (g == 0) {
        if (tid < wa) {
            // PDAMAX returns INDX = IX for a zero maximum (pdamax_.c:486).
            const int p = sl.s_pv[tid];
            ipiv[row0 + tid] = row0 + (p >= 0 ? p : tid) + 1;
            if (p < 0) atomicMin(zero_col, col0 + tid + 1);
        }
        for (int idx = tid; idx < wa * wa; idx += (int)blockDim.x) {
            const int j = idx % wa, c = idx / wa;
            if (c >= j) A[j + (size_t)c * lda] = sl.u[j][(c & 3) * NC + (c >> 2) - (j >> 2)];
        }
    }

    // The leaf's interchanges on the block column's other columns: the
    // lcols columns left of the leaf and the rcols right of it.  Wave 0
    // composes the sequence (j, p_j) into destination <- source row pairs
    // (lane k holds pair k; at most 2 wa <= 64 rows move).  Then every wave
    // rewrites CR columns at a time, lane k moving pair k: the wave's loads
    // of a column all complete before its stores to that column.
    const int ne = lcols + rcols;
    if (ne <= 0) return;
    if (wave == 0) {
        int dst = -1, src = -1, cnt = 0;
        for (int j = 0; j < wa; j++) {
            const int p = sl.s_pv[j];
            if (p == j || p < 0) continue;
            const uint64_t mj = __ballot(dst == j), mp = __ballot(dst == p);
            const int lj = mj ? __ffsll((unsigned long long)mj) - 1 : -1;
            const int lp = mp ? __ffsll((unsigned long long)mp) - 1 : -1;
            const int sj = lj >= 0 ? __shfl(src, lj) : j;  // row now at position j
            const int sp = lp >= 0 ? __shfl(src, lp) : p;  // row now at position p
            if (lj >= 0) { if (lane == lj) src = sp; }
            else { if (lane == cnt) { dst = j; src = sp; } cnt++; }
            if (lp >= 0) { if (lane == lp) src = sj; }
            else { if (lane == cnt) { dst = p; src = sj; } cnt++; }
        }
        if (lane < cnt) { sl.s_dst[lane] = dst; sl.s_src[lane] = src; }
        if (lane == 0) sl.s_npair = cnt;
    }
    __syncthreads();
    if (lane >= sl.s_npair) return;
    constexpr int CR = 8;
    const int rd = sl.s_dst[lane], rs = sl.s_src[lane];
    for (int e0 = (g * nw + wave) * CR; e0 < ne; e0 += G * nw * CR) {
        T v[CR];
#pragma unroll
        for (int c = 0; c < CR; c++) {
            const int e = e0 + c;
            const int cc = (e < lcols) ? (e - lcols) : (wa + e - lcols);
            if (e < ne) v[c] = A[(ptrdiff_t)cc * lda + rs];
        }
#pragma unroll
        for (int c = 0; c < CR; c++) {
            const int e = e0 + c;
            const int cc = (e < lcols) ? (e - lcols) : (wa + e - lcols);
            if (e < ne) A[(ptrdiff_t)cc * lda + rd] = v[c];
        }
    }
}

template <typename T, int NC, int NQ, bool SOLO, int PT, int WPE>
void launch_leaf(T *A, int lda, int m, int wa, int lcols, int rcols, int row0, int col0, int *ipiv,
                 const PanelWork<T> &pw, int threads, int G, LeafPlace place, hipStream_t s)
{
    PanelMailState &ms = *pw.mail_state;
    if (threads > PT) throw std::logic_error("panel leaf: workgroup larger than its kernel's");
    if constexpr (SOLO) {
        // the mailbox and its record stay as the last exchanging launch left them
        hipLaunchKernelGGL((panel_leaf_kernel<T, NC, NQ, true, PT, WPE, false>), dim3(1), dim3(threads), 0,
                           s, A, lda, m, wa, lcols, rcols, row0, col0, ipiv, pw.mail, 0, 0, 0,
                           pw.abort_flag, pw.zero_col, pw.spin_limit, 1, 0, pw.yield, 0u, 0u,
                           (uint64_t)0);
        SLA_LAUNCH_CHECK();
    } else {
        auto go = [&](auto yields, int stride, unsigned yield_id, unsigned after_id) {
            const int first = stride == 1 ? 0 : (int)(ms.launches % XCDS);
            hipLaunchKernelGGL((panel_leaf_kernel<T, NC, NQ, false, PT, WPE, decltype(yields)::value>),
                               dim3(G * stride), dim3(threads), 0, s, A, lda, m, wa, lcols, rcols, row0,
                               col0, ipiv,
                               pw.mail, (int)(ms.launches & 1u), ms.prev_wa, ms.prev_g,
                               pw.abort_flag, pw.zero_col, pw.spin_limit, stride, first, pw.yield,
                               yield_id, after_id, pw.patience);
            SLA_LAUNCH_CHECK();
            ms.launches++;
            ms.prev_wa = wa;
            ms.prev_g = G;
        };
        if (place != LEAF_ONE_XCD_YIELDS) return go(std::false_type(), place == LEAF_SPREAD ? 1 : XCDS, 0u, 0u);
        if constexpr (leaf_may_yield(NC, PT)) {
            if (wa < 2) throw std::logic_error("panel leaf: a leaf of one column cannot give way");
            const unsigned id = std::max(1u, ms.launches + 1);
            go(std::true_type(), XCDS, id, 0u);
            go(std::true_type(), 1, 0u, id);
        } else {
            throw std::logic_error("panel leaf: a leaf of this kind does not give way");
        }
    }
}

// NC: registers per row and lane.
template <typename T, int NC>
void leaf_of_width(T *A, int lda, int m, int wa, int lcols, int rcols, int row0, int col0,
                   int *ipiv, const PanelWork<T> &pw, hipStream_t s)
{
    const LeafPlan p = leaf_plan(m, wa, pw.target_wgs, pw.beside, pw.num_cus == XCDS * XCD_CUS);
    constexpr int V = leaf_values(NC);
    if (p.wgs > LEAF_GMAX)
        throw std::runtime_error("panel leaf: panel too tall for the leaf's workgroup limit");
#define SLA_LEAF(V, SOLO, PTV, WPE)                                                                 \
    launch_leaf<T, NC, (V) / NC, SOLO, PTV, WPE>(A, lda, m, wa, lcols, rcols, row0, col0, ipiv, pw, \
                                                 64 * p.waves, p.wgs, p.place, s)
    if (p.wgs == 1) {
        if (p.values == V) SLA_LEAF(V, true, 512, 4);
        else SLA_LEAF(64, true, 512, 2);
    } else if (p.values != V) SLA_LEAF(64, false, 512, 2);
    else if (p.waves == 4) SLA_LEAF(V, false, 256, 4);
    else SLA_LEAF(V, false, 512, 4);
#undef SLA_LEAF
}

}  // namespace

template <typename T>
unsigned panel_leaf(T *A, int lda, int m, int wa, int lcols, int rcols, int row0, int col0,
                    int *ipiv, const PanelWork<T> &pw, hipStream_t s)
{
    if (wa > 32) throw std::runtime_error("panel leaf: width above 32");
    switch (leaf_nc(wa)) {
    case 2: leaf_of_width<T, 2>(A, lda, m, wa, lcols, rcols, row0, col0, ipiv, pw, s); break;
    case 4: leaf_of_width<T, 4>(A, lda, m, wa, lcols, rcols, row0, col0, ipiv, pw, s); break;
    default: leaf_of_width<T, 8>(A, lda, m, wa, lcols, rcols, row0, col0, ipiv, pw, s);
    }
    return 0;  // the mailbox exchange adds no barrier arrivals
}

// The build compiles this file twice, SLA_PANEL_TYPE = 64 and 32, so that the
// leaf instances of the two storage types build in parallel; without the macro
// both are instantiated here.
#if !defined(SLA_PANEL_TYPE) || SLA_PANEL_TYPE == 64
template unsigned panel_leaf<double>(double *, int, int, int, int, int, int, int, int *,
                                     const PanelWork<double> &, hipStream_t);
#endif
#if !defined(SLA_PANEL_TYPE) || SLA_PANEL_TYPE == 32
template unsigned panel_leaf<float>(float *, int, int, int, int, int, int, int, int *,
                                    const PanelWork<float> &, hipStream_t);
#endif

}  // namespace sla
