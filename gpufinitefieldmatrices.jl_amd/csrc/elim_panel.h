// elim_panel.h -- panel factorisation of the blocked elimination (gfx950).
//
// The panel W[kr0:m, c0:c0+w] (w <= 32) is held in registers, one row per
// lane and one FP64 register pair per column, by as many wavefronts as there
// are 64-row groups.  The pivot rule makes the columns a serial chain (the
// largest residue of column j is known only after the update by pivot
// j - 1), so the kernel is bound by that chain's latency, not by arithmetic
// or bandwidth; everything that is not on the chain runs while the chain
// waits.  One column:
//
//   A  reduce the column, find the wave's best (residue, lowest position) by
//      DPP and publish it;
//   C  (over several workgroups) rebuild the candidate's row, scale it by its
//      inverse and publish it;
//   B  apply the previous pivot to the columns after this one and write its
//      record down;
//   D  find the winner among the waves' candidates;
//   E  take its row (one workgroup: rebuild and scale it now);
//   F  apply the row to the next column, go on.
//
// A row as it is now is rebuilt by left-looking sums, x_j = a_j -
// sum_k l_k u_kj with lane j column j, because nothing cheap moves one lane's
// 32 registers across the lanes: 16 one-lane LDS writes took 480 cycles, more
// with several waves.  Factors reach all lanes by DPP (row_newbcast, 5 cycles
// an FMA; by LDS broadcast or readlane it is 20 to 25).
//
// The column loop is rolled four columns at a time: then the columns move
// four registers down (and the pivots' scaled rows four up), so the code of
// a step runs from the instruction cache; moving them at every column cost
// 250 cycles of a step, unrolling all 32 runs each instruction once, from
// memory.
//
// Up to 256 rows: one workgroup, the candidates meet in LDS behind one
// barrier a column.  More rows: one wave per 64 rows, four to a workgroup,
// on the CUs of ONE XCD, and the candidates meet in that XCD's L2: every
// wave stores its key in its own slot, every lane of every wave polls one
// slot, and no wave ever waits at a barrier.  Every word carries its step's
// tag, so a word is either recognised as old or whole; key slots alternate
// between two sets, and a wave overwrites a set only after every wave has
// published the step in between, that is after every wave has read it.
// Measured (one key and one row exchanged per step, 2 to 32 workgroups): 1490
// cycles with loads that bypass L1 (non-temporal) and plain stores inside one
// XCD, 2050 with agent-scope loads and stores, 2700 to 3100 across XCDs.
//
// The panel also leaves the inverse of its pivot triangle (PanelSolve), from the
// upper half of the waves that rebuild rows, at no step of the chain.
//
// All workgroups have to be on the XCD at once.  The rows' own LDS is 66.6 KB,
// and the scaled rows are int32 there rather than FP64, so that two workgroups
// fit on a CU and 64 (16,384 rows) on an XCD.  (The panel of one workgroup keeps
// FP64: the conversions took 0.5 us of its 33 mod 11.)
//
// A 32-column panel mod 65521 takes 45 us at 4096 rows and 37 us at 256,
// mod 2^26 - 5 51 and 48; at 8192 rows, where every CU has one workgroup, 56
// and 65, with two of them on some or all CUs 66 and 80 at 9000 rows and 76 and
// 89 at 16,384 (before the rows were published scaled, the
// inverses looked up and the records moved off the chain: 50, 38, 60 and 53;
// one 512-thread workgroup with eight rows a thread, unrolled, and the rows
// published by one-lane LDS writes: 94 and 52 mod 65521, as four panels of 8
// columns).  Of a step's 2500 cycles over an XCD about 1100 are the key's way
// there and 400 the row's; on one workgroup it is 1950.
#pragma once
#include <type_traits>

#include "common.h"

namespace {

constexpr int PNW = 32;       // panel columns
constexpr int PWAVES = 4;     // waves of a workgroup, one per SIMD
constexpr int PXS = 256;      // slots of one exchange set (waves of a panel)
constexpr int PINV = 1 << 18;  // entries of the table of small inverses
constexpr int PSINGLE = 64 * PWAVES;  // rows of the one-workgroup panel
constexpr int XCD_CUS = 32;   // CUs of an XCD
constexpr uint32_t PABORT = 0x80000000u;
constexpr uint32_t PUNSCALED = 0x80000000u;  // beside a row's tag: not scaled yet

// compile-time loop: f(integral_constant<int, J>) for J = B .. E-1
template <int B, int E> struct Unroll {
    template <class F> __device__ __forceinline__ static void run(F &f)
    {
        f(std::integral_constant<int, B>{});
        Unroll<B + 1, E>::run(f);
    }
};
template <int E> struct Unroll<E, E> {
    template <class F> __device__ __forceinline__ static void run(F &) {}
};

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

struct PanelCtl {
    int npiv;    // pivots found
    int status;  // 0 all columns consumed, 1 zero column (pluq stop),
                 // 2 rows exhausted, 3 pivot not invertible, 4 not run (an
                 // earlier panel stopped), 5 not run (its workgroups did not
                 // meet on one XCD), 6 an exchange did not end, 7 not run
                 // (no pivot among the first rows, k_panel_any)
    int ncols;   // panel columns consumed
    int nmap;    // entries of the row gather map
    int kr0;     // first row of the panel
};

// exchange area of the panels that span workgroups (device memory, kept in
// the context; every launch uses tags of its own)
struct PanelExchange {
    unsigned long long key[2][PXS];       // residue 26, 32767 - position 15, lane 6, tag 17 bits
    unsigned long long row[2][PXS][2 * PNW];  // entry (signed), 31 bits of tag under PUNSCALED
};

// What a panel leaves for the solves with its pivot rows: the rows of U of any
// other columns are T times the pivot rows' old values.
struct PanelSolve {
    int32_t t[PNW][PNW];  // balanced; row: panel column (0: no pivot), column: pivot
    int32_t num[PNW];     // pivot of a panel column, or -1
};

// a word of host memory that shows the host, still enqueuing, that a panel stopped
__device__ __forceinline__ void tell(int *word)
{
    if (word) __hip_atomic_store(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct PanelArgs {
    int32_t *W;
    int64_t ldw;
    int m, kr0, c0, w, ple, KC, FAR;
    ModP mp;
    const uint32_t *invs;  // inverses of 0..PINV-1 (0: none)
    int32_t *ipiv, *pivval, *pivinv, *pivcol, *map_dst, *map_src, *stage;
    PanelCtl *ctl;
    PanelSolve *solve;
    int *abort, *cursor, *told;
    int strict;          // a column without a pivot raises the abort flag, too
    PanelExchange *x;
    uint32_t *arrive;
    int G;               // workgroups that take part
    uint32_t tag;        // tag of the step before the first
    int *lost;           // raised by a wave whose exchange did not end
    int spins;           // EXCHANGE_SPINS
    long long patience;  // cycles a workgroup waits for the others to start; below 0 none goes on
};

// x mod p for exact integers |x| <= 2^51: fl(x * pinv) is within
// |x| 2^-52 / p <= 1/(2p) of x/p, so q = rint(.) is within 1/2 + 1/(2p) < 1 of
// x/p, r = x - q p is exact with |r| < p, and one fix-up brings it to [0,p).
__device__ __forceinline__ double dmod_near(double x, const ModP &mp)
{
    const double r = fma(-rint(x * mp.pinv), mp.pd, x);
    return r < 0.0 ? r + mp.pd : r;
}

// x - p rint(x/p) for |x| < 2^53 is exact, and at most p/2 + p 2^-22 in
// magnitude (x pinv is off by at most 2^-52 |x|/p).
__device__ __forceinline__ double near_mod(double x, const ModP &mp) { return fma(-rint(x * mp.pinv), mp.pd, x); }
// the residue in [0,p) of a balanced one, and back
__device__ __forceinline__ double from_near(double r, const ModP &mp) { return r < 0.0 ? r + mp.pd : r; }
__device__ __forceinline__ double to_near(double c, const ModP &mp) { return c > (double)mp.half ? c - mp.pd : c; }

__device__ __forceinline__ double readlane_f64(double x, int l)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, l), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sums with a factor from another lane of the row of 16 lanes
// (v_fmac_f64_dpp, row_newbcast), which the compiler does not form by itself.
// The wait states between a vector write of x and its use by DPP are at the
// head of each block.
// v[k] += (x of lane L0 + k) * y for k < N
template <int L0, int N> __device__ __forceinline__ void fmac_lanes(double *v, double x, double y)
{
    static_assert((L0 == 0 && (N == 16 || N == 4)) || (L0 == 2 && N == 14), "the blocks below");
    if constexpr (N == 16) {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %16, %17 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %16, %17 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %16, %17 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %16, %17 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %4, %16, %17 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %5, %16, %17 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %6, %16, %17 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %7, %16, %17 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %8, %16, %17 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %9, %16, %17 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %10, %16, %17 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %11, %16, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %12, %16, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %13, %16, %17 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %14, %16, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %15, %16, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]),
              "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15])
            : "v"(x), "v"(y));
    } else if constexpr (N == 14) {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %14, %15 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %14, %15 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %14, %15 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %14, %15 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %4, %14, %15 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %5, %14, %15 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %6, %14, %15 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %7, %14, %15 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %8, %14, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %9, %14, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %10, %14, %15 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %11, %14, %15 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %12, %14, %15 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %13, %14, %15 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]),
              "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13])
            : "v"(x), "v"(y));
    } else {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %4, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %4, %5 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %4, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])
            : "v"(x), "v"(y));
    }
}
// acc[k] += (x of lane L0 + k) * y[k] for k < 4
template <int L0> __device__ __forceinline__ void dot_lanes(double *acc, double x, const double *y)
{
    asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %4, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
        : "v"(x), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
}

// a^{-1} mod p for a wave-uniform a in [1, p), 0 if it has none.  Extended
// Euclid is a chain of about 15 to 25 divisions on the panel's critical path;
// this looks a up in the table of the inverses below PINV, or p - a, since
// pivots are the largest of many residues.  Only p > PINV leaves anything else:
// then, by Dirichlet's approximation theorem, some multiplier t <= 256 brings
// a t within p/257 < PINV of a multiple of p (every lane tries four), and the
// remainder is looked up.  For a modulus that is not prime a remainder without
// an inverse says nothing about a, and Euclid decides.  With a table of 1024 in
// LDS and one or two such rounds a step spent 540 cycles here mod 65521 and 940
// mod 2^26 - 5; the lookup goes on beside the rebuilding of the row.
template <int MODE> __device__ __forceinline__ uint32_t table_place(uint32_t a, const ModP &mp)
{
    return MODE == 0 || mp.p <= PINV ? a : mp.p32 - a;
}
// the inverse from the table's entry t at a's place, 0 if that has none
template <int MODE> __device__ __forceinline__ uint32_t table_inverse(uint32_t a, uint32_t t, const ModP &mp)
{
    if (MODE == 0 || mp.p <= PINV) return t;
    return mp.p32 - a < (uint32_t)PINV && t != 0 ? mp.p32 - t : 0u;
}
__device__ __forceinline__ uint32_t search_inverse(uint32_t a, const uint32_t *__restrict__ T, const ModP &mp, int lane)
{
    uint32_t inv = 0;
    if (mp.p > PINV) {
        // lane l tries l + 1 + 64 i and keeps the one that comes nearest
        double r = 0.0, t = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double ti = (double)(lane + 1 + 64 * i), x = near_mod((double)a * ti, mp);
            const bool nearer = i == 0 || fabs(x) < fabs(r);
            r = nearer ? x : r;
            t = nearer ? ti : t;
        }
        const int l = (int)__builtin_ctzll(__ballot(fabs(r) * 257.0 <= mp.pd)) & 63;
        r = readlane_f64(r, l);
        t = readlane_f64(t, l);
        const double z = (double)T[(uint32_t)fabs(r) & (PINV - 1)] * (r < 0.0 ? -t : t);
        inv = (uint32_t)uniform((int)(uint32_t)from_near(near_mod(z, mp), mp));
    }
    if (inv == 0) inv = (uint32_t)uniform((int)modinv_fast(a, mp));
    return inv;
}

// The workgroups of a panel meet before anything is written: nobody waits
// for a workgroup that has no CU yet longer than `patience`, and either all go
// on (the count was reached before anyone gave up) or none does.  They also
// have to share an XCD, or the exchange would not see their stores: beside the
// count (bits 0-6) the word sums the XCD numbers (8-16) and their squares
// (17-28), and only equal numbers have both means.
__device__ __forceinline__ uint32_t panel_xcd()
{
    uint32_t x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    return x & 7;
}
__device__ __forceinline__ void panel_arrive(uint32_t *word)
{
    const uint32_t x = panel_xcd();
    atomicAdd(word, 1u + (x << 8) + (x * x << 17));
}
__device__ __forceinline__ bool panel_meet(uint32_t *word, uint32_t G, long long patience)
{
    const uint32_t x = panel_xcd();
    const long long t0 = __builtin_readcyclecounter();
    for (;;) {
        const uint32_t cur = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cur & PABORT) return false;
        if ((cur & 0x7fu) == G && patience >= 0) return cur == G * (1u + (x << 8) + (x * x << 17));
        if ((long long)__builtin_readcyclecounter() - t0 > patience && atomicCAS(word, cur, cur | PABORT) == cur)
            return false;
        __builtin_amdgcn_s_sleep(1);
    }
}

// A word of the exchange, past L1.  The first polls are non-temporal loads
// (they leave nothing in L1); should one ever find an old line, the later ones
// are agent-scope loads.
__device__ __forceinline__ unsigned long long exchange_load(unsigned long long *p, int spins)
{
    asm volatile("" ::: "memory");
    if (spins < 256) return __builtin_nontemporal_load(p);
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void exchange_store(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
constexpr int EXCHANGE_SPINS = 1 << 20;  // looks at a word before its step counts as lost

// Arithmetic of a panel by the modulus.  The columns are exact integers in
// FP64 and one FMA applies a pivot; multipliers and scaled rows are balanced
// (|x| <= h = p/2, in mode 2 up to h + 8):
//   0  p < 2^16, and
//   1  p <= 2^24: 31 products below 2^46 stay below 2^51;
//   2  p <= 2^26: reduced after at most five products (< 2^53).

// wave64 maximum: DPP within the rows of 16 lanes, then from row to row (each
// step takes two wait states and one instruction; the last lane has it all)
__device__ __forceinline__ uint32_t wave_max_dpp(uint32_t v)
{
    v = kmax(v, dpp32<0xB1>(v));   // quad_perm [1,0,3,2]
    v = kmax(v, dpp32<0x4E>(v));   // quad_perm [2,3,0,1]
    v = kmax(v, dpp32<0x141>(v));  // row_half_mirror
    v = kmax(v, dpp32<0x140>(v));  // row_mirror
    v = kmax(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = kmax(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The best of the lanes' (residue, 32767 - position): residue << 15 | the
// latter, wave-uniform, and a lane that has it.  Below 2^16 both share a word.
// Above, ties are rare: the positions are compared only when there is one.
template <int MODE> __device__ __forceinline__ uint64_t panel_best(uint32_t v, uint32_t notpos, int *lane_of)
{
    if (MODE == 0) {
        const uint32_t k = (v << 15) | notpos, top = wave_max_dpp(k);
        *lane_of = (int)__builtin_ctzll(__ballot(k == top));
        return top;
    }
    const uint32_t top = wave_max_dpp(v);
    uint64_t at = __ballot(v == top);
    if (at & (at - 1)) {
        const uint32_t np = wave_max_dpp(v == top ? notpos : 0u);
        at = __ballot(v == top && notpos == np);
    }
    const int l = (int)__builtin_ctzll(at);
    *lane_of = l;
    return ((uint64_t)top << 15) | (uint32_t)__builtin_amdgcn_readlane((int)notpos, l);
}

template <bool MULTI, int MODE>
__global__ __launch_bounds__(64 * PWAVES, MULTI ? 2 : 1) void k_panel(PanelArgs a)
{
    typedef unsigned long long u64;
    int rank = 0;
    if (MULTI) {
        // workgroups are dealt to the XCDs in turn: every eighth lands on the
        // same one
        if (blockIdx.x & 7) return;
        rank = blockIdx.x >> 3;
    }
    const ModP mp = a.mp;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    if (a.abort && *a.abort) {
        // an earlier panel of this block stopped, or this one's workgroups
        // gave up before this one started
        if (rank == 0 && tid == 0) {
            const bool gave_up =
                MULTI && (__hip_atomic_load(a.arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & PABORT);
            *a.ctl = PanelCtl{0, gave_up ? 5 : 4, 0, 0, a.kr0};
        }
        return;
    }
    // the first row comes from the device cursor when the previous panel's
    // pivot count is not known to the host (lu, rref)
    const int kr0 = uniform(a.cursor ? *a.cursor : a.kr0);

    // original and reduced columns by local row, a wave's rows of 64 (the odd
    // pitch spreads a row of the panel over the banks)
    __shared__ int32_t s_A[PWAVES][PNW][65], s_L[PWAVES][PNW][65];
    // scaled rows (negated, balanced) by column, and the rows of T
    typedef std::conditional_t<MULTI, int32_t, double> scaled_t;
    __shared__ scaled_t s_U[PNW][2 * PNW];
    __shared__ __attribute__((aligned(16))) double s_key[2][PWAVES];
    __shared__ int s_go;

    if (MULTI && tid == 0) panel_arrive(a.arrive);
    const int w = a.w, rows = a.m - kr0, gw = rank * PWAVES + wave, nw = MULTI ? a.G * PWAVES : PWAVES;
    const int i = gw * 64 + lane;  // panel row of this lane
    const bool exists = i < rows;
    const int64_t ldw = a.ldw;
    int32_t *const Wp = a.W + (int64_t)a.c0 * ldw;  // panel columns
    // register k holds column 4 * chunk + k (the last ones are never used as
    // columns)
    constexpr int NV = PNW + 4;
    double v[NV];
    {
        const uint32_t r = (uint32_t)min(kr0 + i, a.m - 1);
        const int32_t *col = Wp;
        int32_t x[PNW];
#pragma unroll
        for (int j = 0; j < PNW; ++j) {
            x[j] = col[r];
            col += j + 1 < w ? ldw : 0;
        }
#pragma unroll
        for (int j = 0; j < PNW; ++j) {
            s_A[wave][j][lane] = x[j];
            v[j] = exists ? (double)x[j] : 0.0;
        }
#pragma unroll
        for (int j = PNW; j < NV; ++j) v[j] = 0.0;
    }
    // every row is in registers before its wave publishes a key, and no wave
    // stores to W before it has every wave's last key
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (MULTI) {
        if (tid == 0) s_go = panel_meet(a.arrive, (uint32_t)a.G, a.patience);
        __syncthreads();
        if (!s_go) {
            if (tid == 0) {
                __threadfence();
                *a.abort = 1;
                if (rank == 0) *a.ctl = PanelCtl{0, 5, 0, 0, kr0};
            }
            return;
        }
    }

    // position of the row now (rows that are not pivots: pc or more); the pivot
    // that moved it last
    int pos = exists ? i : -1, dk = 0;
    int pc = 0, status = 0, consumed = w, spins = 0;
    uint32_t pivcols = 0;  // columns that have a pivot
    // lane t: pivot t's old position, value, inverse and column; the position
    // again, or -1 when a later pivot came from there, too
    int ip_l = -1, pv_l = 0, pi_l = 0, pj_l = 0, iq_l = -1;
    bool active = true;
    // the previous pivot: this row's multiplier and the scaled row (both
    // negated), and what is still to be written down of it
    double nl = 0.0, nup = 0.0;
    int Ipp = -2, atp = -2, Vp = 0;
    auto write_down = [&](int jc) __attribute__((always_inline)) {
        s_U[jc & (PNW - 1)][lane] = (scaled_t)nup;
        iq_l = iq_l == Ipp ? -1 : iq_l;
        const bool here = lane == atp;
        ip_l = here ? Ipp : ip_l;
        iq_l = here ? Ipp : iq_l;
        pv_l = here ? Vp : pv_l;
        // the identity's own column of the scaled row is the pivot's inverse
        const double iv = -readlane_f64(nup, (PNW + jc) & 63);
        pi_l = here ? (int)from_near(iv, mp) : pi_l;
        pj_l = here ? jc : pj_l;
        atp = Ipp = -2;
    };
    // the negated scaled rows, lane j column j, lane 32 + j column j of T, zero
    // where a column has no pivot: column jc of the running chunk in h[3 - jc % 4], older ones
    // from h[4] on
    constexpr int NH = PNW + 4;
    double h[NH];
#pragma unroll
    for (int k = 0; k < NH; ++k) h[k] = 0.0;
    const int back = lane & 15, col = lane & (PNW - 1);
    // columns 4 c .. 4 c + 3; HW: earlier columns there may be, CW: columns after
    // the current one (in 16s or 4s over 16)
    auto chunk = [&](int c, auto HWC, auto CWC) __attribute__((always_inline)) {
        constexpr int HW = decltype(HWC)::value, CW = decltype(CWC)::value;
        auto step = [&](auto SC) __attribute__((always_inline)) {
            constexpr int s = decltype(SC)::value, par = s & 1;
            const int jc = 4 * c + s;
            // A: column jc is final.  Below 2^51 the residue comes without a
            // fix-up: (x + 1/2) / p is at least 1/(2p) away from every integer,
            // and its rounded product is nearer to it than that
            double cn;
            uint32_t ci;
            if constexpr (MODE == 2) {
                cn = near_mod(v[s], mp);
                ci = (uint32_t)from_near(cn, mp);
            } else {
                const double r = fma(-floor(fma(v[s], mp.pinv, 0.5 * mp.pinv)), mp.pd, v[s]);
                ci = (uint32_t)r;
                cn = MODE == 0 ? r : to_near(r, mp);
            }
            s_L[wave][jc][lane] = (int32_t)ci;
            active = active && jc < w;
            if (active && pc >= rows) {
                status = 2;
                consumed = jc;
                active = false;
            }
            const uint32_t tag = (a.tag + 1 + (uint32_t)jc) & 0x7fffffffu, tag17 = tag & 0x1ffffu;
            // local row lr of wave lw as it is now, lane j column j, from its
            // original entries and multipliers (h is zero where there are
            // none); below 2^16 the sums stay below 2^37 and the
            // multipliers need not be balanced.  Lanes 32 + j hold the same
            // for the columns of an identity beside the panel, which turn
            // into the rows of T: the upper half of the wave is free
            auto row_now = [&](int lw, int lr) __attribute__((always_inline)) {
                double x[4] = {lane < PNW ? (double)s_A[lw][col][lr] : (col == jc ? 1.0 : 0.0), 0.0, 0.0, 0.0};
                double l0 = (double)s_L[lw][max(jc - 1 - back, 0)][lr], l1 = 0.0;
                if (HW > 16) l1 = (double)s_L[lw][max(jc - 17 - back, 0)][lr];
                if (MODE != 0) {
                    l0 = to_near(l0, mp);
                    l1 = to_near(l1, mp);
                }
                auto dot = [&](auto KC) __attribute__((always_inline)) {
                    constexpr int k = 4 * decltype(KC)::value;
                    dot_lanes<k & 15>(x, k < 16 ? l0 : l1, h + 4 - s + k);
                    if constexpr (MODE == 2 && (k & 15) == 12)
#pragma unroll
                        for (int q = 0; q < 4; ++q) x[q] = near_mod(x[q], mp);
                };
                Unroll<0, HW / 4>::run(dot);
                return (x[0] + x[1]) + (x[2] + x[3]);
            };
            // a row as the pivot's: scaled by its inverse, negated, balanced
            auto scaled = [&](double x, uint32_t inv) __attribute__((always_inline)) {
                const double xi = MODE == 0 ? x * (double)inv : near_mod(x, mp) * to_near((double)inv, mp);
                return near_mod(-xi, mp);
            };
            // B: the previous pivot on the columns after this one (register k is
            // k - s + 1 columns after it), its row by the distance from this one
            double u0 = 0.0, u1 = 0.0;
            auto fetch_row = [&]() __attribute__((always_inline)) {
                const uint64_t b = __builtin_bit_cast(uint64_t, -nup);
                auto column = [&](int j) {
                    const int src = 4 * (jc - 1 + j);
                    const uint32_t lo = __builtin_amdgcn_ds_bpermute(src, (int)(uint32_t)b);
                    const uint32_t hi = __builtin_amdgcn_ds_bpermute(src, (int)(uint32_t)(b >> 32));
                    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
                };
                u0 = column(back);
                u1 = column(16 + back);
            };
            auto apply_row = [&]() __attribute__((always_inline)) {
                fmac_lanes<2, 14>(v + s + 1, u0, nl);
                fmac_lanes<0, CW>(v + s + 15, u1, nl);
                if constexpr (MODE == 2 && s == 3) {
#pragma unroll
                    for (int k = s + 1; k < (CW == 16 ? PNW : 19); ++k) v[k] = near_mod(v[k], mp);
                }
                write_down(jc - 1);
            };
            double nu = 0.0, un = 0.0;  // the scaled row (negated); its next column
            if (!active) {
                fetch_row();
                apply_row();
            } else {
                const bool alive = pos >= pc;
                int cl;
                const uint64_t mine = panel_best<MODE>(alive ? ci : 0u, alive ? 0x7fffu - (uint32_t)pos : 0u, &cl);
                if (MULTI) {
                    if (lane == 0) exchange_store(&a.x->key[par][gw], (mine << 23) | ((uint32_t)cl << 17) | tag17);
                } else {
                    if (lane == 0) s_key[par][wave] = __builtin_bit_cast(double, (mine << 8) | (uint32_t)(wave * 64 + cl));
                }
                // the table's entry for this wave's candidate, in case it wins
                const uint32_t early = a.invs[min(table_place<MODE>((uint32_t)(mine >> 15), mp), (uint32_t)PINV - 1)];
                fetch_row();
                uint64_t best;
                int at;  // MULTI: winner's slot, else its local row
                if (MULTI) {
                    // C: the first look at the keys goes out before the row, or it
                    // would wait for that store to end
                    const double x = row_now(wave, cl);
                    const uint32_t inv = table_inverse<MODE>((uint32_t)(mine >> 15), early, mp);
                    const int32_t xi = (int32_t)(inv != 0 ? scaled(x, inv) : near_mod(x, mp));
                    u64 t = exchange_load(&a.x->key[par][min(lane, nw - 1)], 0);
                    asm volatile("" ::: "memory");
                    exchange_store(&a.x->row[par][gw][lane],
                                   ((u64)(uint32_t)xi << 32) | tag | (inv != 0 ? 0u : PUNSCALED));
                    apply_row();
                    // D
                    u64 kt = 0;
                    int slot = 0;
                    for (int b = 0; b < nw; b += 64) {
                        const int idx = min(b + lane, nw - 1);
                        if (b != 0) t = exchange_load(&a.x->key[par][idx], spins);
                        while (!__all((uint32_t)(t & 0x1ffffu) == tag17)) {
                            if (++spins > a.spins) break;
                            t = exchange_load(&a.x->key[par][idx], spins);
                        }
                        if (t > kt || b == 0) {
                            kt = t;
                            slot = idx;
                        }
                    }
                    int l;
                    best = panel_best<MODE>((uint32_t)(kt >> 38), (uint32_t)(kt >> 23) & 0x7fffu, &l);
                    at = __builtin_amdgcn_readlane(slot, l);
                } else {
                    apply_row();
                    __syncthreads();
                    // words below 2^49 compare as the (denormal) doubles they spell
                    const uint64_t k = __builtin_bit_cast(uint64_t, fmax(fmax(s_key[par][0], s_key[par][1]),
                                                                        fmax(s_key[par][2], s_key[par][3])));
                    const uint32_t lo = uniform((int)(uint32_t)k), hi = uniform((int)(uint32_t)(k >> 32));
                    best = (((u64)hi << 32) | lo) >> 8;
                    at = (int)(lo & 0xffu);
                }
                // E: the scaled row
                const uint32_t V = (uint32_t)(best >> 15);
                bool piv = V != 0;
                if (MULTI) {
                    u64 *rp = &a.x->row[par][at][lane];
                    u64 t = exchange_load(rp, 0);
                    while (piv && !__all((((uint32_t)t ^ tag) & ~PUNSCALED) == 0)) {
                        if (++spins > a.spins) break;
                        t = exchange_load(rp, spins);
                    }
                    nu = (double)(int32_t)(t >> 32);
                    const bool unscaled = __any((uint32_t)t & PUNSCALED);
                    if (__builtin_expect(!piv || unscaled || spins > a.spins, 0)) {
                        const uint32_t inv = piv && spins <= a.spins ? search_inverse(V, a.invs, mp, lane) : 0u;
                        nu = scaled(nu, inv);
                        piv = inv != 0;
                    }
                } else {
                    asm volatile("" ::"v"(early));
                    const uint32_t entry = a.invs[min(table_place<MODE>(V, mp), (uint32_t)PINV - 1)];
                    const double x = row_now(at >> 6, at & 63);
                    uint32_t inv = (uint32_t)uniform((int)table_inverse<MODE>(V, entry, mp));
                    if (__builtin_expect(inv == 0 || !piv, 0)) {
                        inv = piv ? search_inverse(V, a.invs, mp, lane) : 0u;
                        piv = inv != 0;
                    }
                    nu = scaled(x, inv);
                }
                if (__builtin_expect(!piv, 0)) {
                    const bool lost = spins > a.spins;
                    if (V != 0 || !a.ple || lost) {
                        // a zero column (lu and rref skip it, pluq stops), or no inverse
                        status = lost ? 6 : V == 0 ? 1 : 3;
                        consumed = jc;
                        active = false;
                    }
                }
                spins = 0;
                // F: without a pivot the row is zero and no position matches
                nu = piv ? nu : 0.0;
                un = -readlane_f64(nu, (jc + 1) & 31);
                // the winner moves to pc, the row at pc to Ip
                Ipp = piv ? 0x7fff - (int)(best & 0x7fffu) : -2;
                atp = piv ? pc : -2;
                const bool out = pos == atp;
                dk = out ? pc : dk;
                pos = pos == Ipp ? pc : (out ? Ipp : pos);
                Vp = (int)V;
                pivcols |= piv ? 1u << jc : 0u;
                pc += piv ? 1 : 0;
                nl = pos >= pc ? -cn : 0.0;
            }
            v[s + 1] = fma(nl, un, v[s + 1]);
            nup = nu;
            h[3 - s] = nu;
        };
        Unroll<0, 4>::run(step);
#pragma unroll
        for (int k = 0; k + 4 < NV; ++k) v[k] = v[k + 4];
#pragma unroll
        for (int k = (HW > 16 ? NH : 20) - 1; k >= 4; --k) h[k] = h[k - 4];
    };
    const int chunks = (w + 3) / 4;
    for (int c = 0; c < min(chunks, 4); ++c)
        chunk(c, std::integral_constant<int, 16>{}, std::integral_constant<int, 16>{});
    for (int c = 4; c < chunks; ++c)
        chunk(c, std::integral_constant<int, 32>{}, std::integral_constant<int, 4>{});
    write_down(4 * chunks - 1);

    const int pj_q = __shfl(pj_l, col);  // lanes t and 32 + t: column of pivot t
    // the pivots' scaled rows at their final places, T and the pivots' records,
    // by the first workgroup (every wave has written all of s_U)
    if (rank == 0) {
        int32_t *const dst = Wp + (int64_t)col * ldw + kr0;
        constexpr int RPW = PNW / PWAVES;
        int32_t y[RPW];
#pragma unroll
        for (int q = 0; q < RPW; ++q) y[q] = (int32_t)s_U[wave + PWAVES * q][lane < PNW ? lane : PNW + pj_q];
#pragma unroll
        for (int q = 0; q < RPW; ++q) {
            const int jc = wave + PWAVES * q, t = __popc(pivcols & ((1u << jc) - 1u));
            const bool piv = (pivcols >> jc) & 1u;
            if (lane >= PNW) a.solve->t[jc][col] = piv && col < pc ? -y[q] : 0;
            else if (piv && lane > jc && lane < w) dst[t] = y[q] > 0 ? (int32_t)mp.p32 - y[q] : -y[q];
        }
        if (wave == 0 && lane < PNW)
            a.solve->num[lane] = ((pivcols >> lane) & 1u) ? (int)__popc(pivcols & ((1u << lane) - 1u)) : -1;
        if (wave == 0 && lane < pc) {
            a.ipiv[kr0 + lane] = kr0 + ip_l;
            a.pivval[kr0 + lane] = pv_l;
            a.pivinv[kr0 + lane] = pi_l;
            a.pivcol[kr0 + lane] = a.c0 + pj_l;
        }
    }
    // Row gather map: the pivots in order, then every other row that moved, in
    // the order of the pivots that moved them last: the row that pivot t moved
    // is still where that pivot came from unless a later one came from there
    const int pk = exists && pos < pc ? pos : -1;  // its pivot, if the row is one
    const bool moved = pk >= 0 || (exists && pos != i);
    const uint32_t mask = (uint32_t)__ballot(lane < pc && iq_l >= pc);
    const int e = pk >= 0 ? pk : pc + (int)__popc(mask & ((1u << dk) - 1u));
    const int jp = __shfl(pj_l, max(pk, 0)), jk = pk >= 0 ? jp : PNW;
    if (moved) {
        a.map_dst[e] = kr0 + pos;
        a.map_src[e] = kr0 + i;
    }
    // The old values of every moved row in the block's other columns go to
    // the stage for the update kernel (stage[e + 64 ci], ci counting the block
    // columns left of the panel, then those right of it; both counts are
    // multiples of 32 but in a block's or the matrix's last panel); every row
    // goes to its final position: the multipliers, and at a pivot 1 (the rest
    // of its row is there already).  All loads are issued before any store.
    const int nleft = a.c0 - a.KC, nother = (a.FAR - a.KC) - w;
    const bool some = nother > 0 && __any(moved);
    const uint32_t from = (uint32_t)(kr0 + (moved ? i : 0));
    auto stage_cols = [&](auto NC, int c, int32_t *x) __attribute__((always_inline)) {
        const int32_t *src = a.W + (int64_t)(c < nleft ? a.KC + c : a.KC + c + w) * ldw;
#pragma unroll
        for (int k = 0; k < decltype(NC)::value; ++k) {
            x[k] = src[from];
            src += ldw;
        }
    };
    typedef std::integral_constant<int, 32> N32;
    const bool whole = w == PNW && (nleft & 31) == 0 && nother == 96;  // three full panels beside this one
    int32_t x0[32], x1[32], x2[32];
    if (some && whole) {
        stage_cols(N32{}, 0, x0);
        stage_cols(N32{}, 32, x1);
        stage_cols(N32{}, 64, x2);
    }
    {
        int32_t y[PNW];
#pragma unroll
        for (int j = 0; j < PNW; ++j) y[j] = s_L[wave][j][lane];
        int32_t *dst = Wp;
        const uint32_t to = (uint32_t)(kr0 + pos);
        if (w == PNW && __all(exists && pk < 0)) {
#pragma unroll
            for (int j = 0; j < PNW; ++j) {
                dst[to] = y[j];
                dst += ldw;
            }
        } else if (exists) {
#pragma unroll
            for (int j = 0; j < PNW; ++j) {
                if (j < w && j <= jk) dst[to] = j == jk ? 1 : y[j];
                dst += ldw;
            }
        }
    }
    if (some && moved) {
        int32_t *dst = a.stage + e;
        if (whole) {
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                dst[64 * k] = x0[k];
                dst[64 * (k + 32)] = x1[k];
                dst[64 * (k + 64)] = x2[k];
            }
        } else {
            for (int c = 0; c < nother; ++c)
                dst[64 * c] = a.W[from + (int64_t)(c < nleft ? a.KC + c : a.KC + c + w) * ldw];
        }
    }
    // A wave that misses a step publishes nothing more, so the others miss the
    // next one; but after the last step only the wave itself knows.  Its rows
    // are wrong then: the whole elimination starts again from its input.
    if (MULTI && status == 6 && lane == 0) {
        *a.lost = 1;
        *a.abort = 1;
    }
    if (gw == 0 && lane == 0) {
        *a.ctl = PanelCtl{pc, status, consumed, pc + (int)__popc(mask), kr0};
        if (a.cursor) *a.cursor = kr0 + pc;
        if (a.abort && (status != 0 || (a.strict && pc < w))) {
            *a.abort = 1;
            tell(a.told);
        }
    }
}

// Panel of a reduction whose result does not depend on the pivots (reduced
// echelon form and inverse, prime modulus): any nonzero entry will do, so the
// first 64 rows are enough and no other row is looked at.  One workgroup, a
// row per lane, eight columns per wave, Gauss-Jordan in place without
// divisions: every row but the pivot's becomes V row - m (pivot row), and the
// column is replaced by the identity's, so what is left is A11^{-1} of the
// pivot rows up to a factor per row, whose inverses are taken at the end, all
// at once.  A11^{-1} serves as T and the panel's columns stay as they are: the
// updates subtract A21 (A11^{-1} A12) instead of L21 U12 with L21 = A21 U11^{-1},
// so rows below are never touched here.  The panel's part of U is the identity.
//
// It is bound by its chain: per column one LDS word a row, a barrier, and 40
// FP64 instructions; the next column is updated and passed on before the
// others, some of which wait until the next barrier is behind.  A 32-column
// panel takes 14.3 us mod 65521 and 15.2 us mod 2^26 - 5, whatever its rows (15.0
// and 16.0 with all of them before the barrier; two thirds of it is the chain),
// against 44 and 53 of the general panel over an XCD.  When it came in, RREF of
// 4096^2 and rank 3000 went from 8.2 to 5.1 ms, and with the identity beside the
// matrix in place of L^{-1}, the inverse of 1500^2 mod 2^26 - 5 from 4.0 to 1.94 ms.
// A column without a nonzero entry among the 64 rows says nothing about the rows
// below: status 7, nothing written, and the general panel takes the block.
struct PanelAnyArgs {
    int32_t *W;
    int64_t ldw;
    int m, kr0, c0, w, KC, FAR;
    ModP mp;
    const uint32_t *invs;
    int32_t *ipiv, *pivcol, *map_dst, *map_src, *stage;
    PanelCtl *ctl;
    PanelSolve *solve;
    int *abort, *told;
};
constexpr int PAC = PNW / PWAVES;               // panel columns of a wave
constexpr int PAB = 3;                          // columns updated before a step's barrier, the rest after it
constexpr int PAO = (128 - PNW) / PWAVES;       // other columns of the block, at most

__global__ __launch_bounds__(64 * PWAVES) void k_panel_any(PanelAnyArgs a)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    if (*a.abort) {
        if (tid == 0) *a.ctl = PanelCtl{0, 4, 0, 0, a.kr0};
        return;
    }
    __shared__ double s_col[2][64];
    __shared__ int s_vac[64];
    const ModP mp = a.mp;
    const int w = a.w, kr0 = a.kr0;
    const bool exists = kr0 + lane < a.m;
    const int64_t ldw = a.ldw;
    const uint32_t r = (uint32_t)min(kr0 + lane, a.m - 1);
    const int nleft = a.c0 - a.KC, nother = (a.FAR - a.KC) - w;
    int32_t x[PAC], o[PAO];
#pragma unroll
    for (int k = 0; k < PAC; ++k) x[k] = a.W[r + (int64_t)(a.c0 + min(PAC * wave + k, w - 1)) * ldw];
    // the old values of the other columns, for the stage
    if (nother > 0)
#pragma unroll
        for (int k = 0; k < PAO; ++k) {
            const int c = min(PAO * wave + k, nother - 1);
            o[k] = a.W[r + (int64_t)(c < nleft ? a.KC + c : a.KC + c + w) * ldw];
        }
    double v[PAC];
#pragma unroll
    for (int k = 0; k < PAC; ++k) v[k] = (double)(x[k] > mp.half ? x[k] - (int32_t)mp.p : x[k]);
    uint64_t cand = __ballot(exists);  // rows that are not pivots
    int pk = -1;                       // pivot that this row is
    double d = 1.0, S = 1.0;           // the factor of this row; of the rows that are no pivots yet
    if (wave == 0) s_col[0][lane] = v[0];
    __syncthreads();
    int done = 0;
    double mult = s_col[0][lane];
    for (int ow = 0; ow < PWAVES; ++ow) {
        auto step = [&](auto SC) __attribute__((always_inline)) {
            constexpr int s = decltype(SC)::value, nx = (s + 1) % PAC;
            const int jc = PAC * ow + s;
            if (done != jc || jc >= w) return;  // uniform over the workgroup
            const uint64_t at = __ballot(mult != 0.0) & cand;
            if (at == 0) return;
            const int l = (int)__builtin_ctzll(at);
            cand &= ~(1ull << l);
            const bool pivot = lane == l;
            const double V = readlane_f64(mult, l);
            if (wave == ow) v[s] = pivot ? S : 0.0;
            // products of balanced residues below 2^50 + 2^30, their difference below 2^52
            const double f = pivot ? 1.0 : V, g = pivot ? 0.0 : -mult;
            auto one = [&](int k) __attribute__((always_inline)) {
                v[k] = near_mod(fma(g, readlane_f64(v[k], l), f * v[k]), mp);
            };
            one(nx);
            if (wave == (s + 1 == PAC ? ow + 1 : ow)) s_col[(s + 1) & 1][lane] = v[nx];
            // the other columns while the next one is on its way
#pragma unroll
            for (int k = 1; k <= PAB; ++k) one((nx + k) % PAC);
            __syncthreads();
            mult = s_col[(s + 1) & 1][lane];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = PAB + 1; k < PAC; ++k) one((nx + k) % PAC);
            d = pivot ? V : near_mod(d * V, mp);
            S = near_mod(S * V, mp);
            pk = pivot ? jc : pk;
            done = jc + 1;
        };
        Unroll<0, PAC>::run(step);
    }
    if (done < w) {
        if (tid == 0) {
            *a.ctl = PanelCtl{0, 7, 0, 0, kr0};
            *a.abort = 1;
            tell(a.told);
        }
        return;
    }
    // 1/d: from the table, or d^(p-2)
    double inv;
    {
        const uint32_t dr = (uint32_t)from_near(pk >= 0 ? d : 1.0, mp);
        if (mp.p <= PINV) {
            inv = (double)a.invs[dr];
        } else {
            double b = pk >= 0 ? d : 1.0;
            inv = 1.0;
            for (uint32_t e = mp.p32 - 2; e != 0; e >>= 1) {
                if (e & 1) inv = near_mod(inv * b, mp);
                b = near_mod(b * b, mp);
            }
        }
        inv = to_near(from_near(inv, mp), mp);
    }
    for (int i = tid; i < PNW * PNW; i += 64 * PWAVES)
        if (i / PNW >= w) a.solve->t[i / PNW][i % PNW] = 0;
    if (pk >= 0)
#pragma unroll
        for (int k = 0; k < PAC; ++k)
            a.solve->t[pk][PAC * wave + k] = PAC * wave + k < w ? (int32_t)near_mod(v[k] * inv, mp) : 0;
    // the pivots go to the first w rows, the rows there that are none to the
    // pivots' places
    const bool vacated = pk >= 0 && lane >= w, moves = pk < 0 && lane < w;
    const uint64_t below = (1ull << lane) - 1, mask = __ballot(moves);
    const int rank_v = (int)__popcll(__ballot(vacated) & below), rank_m = (int)__popcll(mask & below);
    if (wave == 0 && vacated) s_vac[rank_v] = lane;
    __syncthreads();
    const int pos = pk >= 0 ? pk : moves ? s_vac[rank_m] : lane;
    const int e = pk >= 0 ? pk : w + rank_m;
    const bool moved = pk >= 0 || moves;
    if (moved) {
#pragma unroll
        for (int k = 0; k < PAC; ++k) {
            const int j = PAC * wave + k;
            if (j < w) a.W[kr0 + pos + (int64_t)(a.c0 + j) * ldw] = pk >= 0 ? (j == pk ? 1 : 0) : x[k];
        }
#pragma unroll
        for (int k = 0; k < PAO; ++k)
            if (PAO * wave + k < nother) a.stage[e + 64 * (PAO * wave + k)] = o[k];
        if (wave == 0) {
            a.map_dst[e] = kr0 + pos;
            a.map_src[e] = kr0 + lane;
        }
    }
    if (wave == 0) {
        if (lane < PNW) a.solve->num[lane] = lane < w ? lane : -1;
        if (lane < w) {  // (nobody reads the pivots' values here, and no swaps)
            a.ipiv[kr0 + lane] = kr0 + lane;
            a.pivcol[kr0 + lane] = a.c0 + lane;
        }
        if (lane == 0) *a.ctl = PanelCtl{w, 0, w, w + (int)__popcll(mask), kr0};
    }
}

}  // namespace
