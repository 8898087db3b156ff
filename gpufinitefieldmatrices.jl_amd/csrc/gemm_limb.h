// gemm_limb.h -- limb form of the mod-p GEMM (gfx950 int8 MFMA).
//
// Each residue r in [0,p) is written in balanced base 256,
// r == sum_u d_u 256^u (mod p), with signed digits d_u in [-128,127] held in
// int8; L = ceil(log256 p) digits (p <= 256^L) cover every residue class.
// The L*L digit products run on v_mfma_i32_32x32x32_i8 with int32
// accumulation, products of equal shift s+t sharing one accumulator; K is cut
// into chunks so that no int32 partial sum can overflow; the 2L-1 shift sums
// are reduced mod p and recombined with weights 256^u mod p in FP64.
//
// The kernel templates live here; gemm_limb_l{1,2,3,4}.hip instantiate the
// launchers for one digit count each (parallel compilation).
#pragma once
#include <type_traits>

#include "common.h"

typedef int v4i __attribute__((ext_vector_type(4)));

// K slicing of one launch: S slices of kslice each; slice s writes at
// C + s*cslice
struct Slices {
    int S = 1;
    int64_t kslice = 0;
    int64_t cslice = 0;
};

struct LimbW {
    double w[7];  // 256^u mod p, balanced (magnitude at most p/2)
    int lazy;     // the recombination of this K chunk is exact without reducing
                  // the digit sums first (limb_lazy)
};

// Recombination of the digit sums, sum_u acc_u w_u.  Shift u collects
// min(u + 1, 2L - 1 - u) digit products of magnitude 2^14 per k, so for k up
// to `kc` the sum is below kc 2^14 (1 + (p/2) sum_{u > 0} pairs(u)); under 2^51
// it is exact in FP64 as it stands (two digits: always; three: k < 4096 at
// 2^23).  Otherwise every digit sum is reduced to a balanced residue first:
// 7 products of at most (2^25 + 1)^2 stay below 2^53.
static inline int limb_lazy(int L, int64_t kc, int64_t p)
{
    double pairs = 0.0;
    for (int u = 1; u < 2 * L - 1; ++u) pairs += u + 1 < 2 * L - 1 - u ? u + 1 : 2 * L - 1 - u;
    return (double)kc * 16384.0 * (1.0 + pairs * (double)(p / 2 + 1)) < 2251799813685248.0;
}

// Launch the limb core for L digits on planes Al (Mp x Kp per digit) and Bl
// (Np x Kp per digit) with a tile_m x tile_n output tile; defined for
// L = 1..4 in gemm_limb_l<L>.hip.
template <int L>
int launch_limb_impl(modp_ctx *ctx, const GemmArgs &g, int epi, const int8_t *Al, int64_t Mp, const int8_t *Bl,
                     int64_t Np, int64_t Kp, const LimbW &lw, int tile_m, int tile_n, const Slices &sl);

namespace {

constexpr int LBK = 64;  // k per MFMA / LDS stage

// Balanced base-256 digits of a residue.  top = 127*(256^L-1)/255: residues
// above it are taken as r - p, which lies in [-128*(256^L-1)/255, -1] because
// p <= 256^L, so L signed digits represent it exactly.
__device__ __forceinline__ int32_t digit_rep(uint32_t r, int32_t top, const ModP &mp)
{
    int32_t x = (int32_t)r;
    return x > top ? x - (int32_t)mp.p32 : x;
}
__device__ __forceinline__ int32_t next_digit(int32_t &x)
{
    const int32_t d = (int32_t)(int8_t)(x & 255);
    x = (x - d) >> 8;
    return d;
}

// The digit planes of both operands in one launch: workgroups [0, na) split A
// (m x k col-major -> Al[s][row][kk], row-major per digit, k contiguous,
// zero-padded to Mp x Kp) by 64 x 64 tiles transposed through LDS, the others
// B (k x n col-major -> Bl[s][col][kk], zero-padded to Np x Kp; k is
// contiguous in memory already), 1024 groups of four k each.  Bound by
// memory: every thread has its sixteen loads in flight before it uses one
// (at indices clamped into the operand, masked afterwards, so that edge
// tiles wait no more than inner ones).  One launch instead of two:
// 5.9 + 4.2 us -> 6.1 us at 1024^2 float64 with two digits, 16.6 + 7.0 -> 12 us at
// 2501 x 1777 and 1777 x 1203 with three.
template <typename T, int L>
__global__ __launch_bounds__(256) void k_split_ab(int64_t m, int64_t n, int64_t k, const T *__restrict__ A, int64_t lda,
                                                  const T *__restrict__ B, int64_t ldb, int8_t *__restrict__ Al,
                                                  int64_t Mp, int8_t *__restrict__ Bl, int64_t Np, int64_t Kp,
                                                  unsigned na, ModP mp, const int *__restrict__ skip)
{
    if (skip && *skip) return;
    constexpr int32_t TOP = (int32_t)(127 * ((((int64_t)1) << (8 * L)) - 1) / 255);
    const int tid = threadIdx.x;
    T x[16];
    if (blockIdx.x < na) {
        __shared__ int32_t tile[64][65];
        const unsigned kt = (unsigned)(Kp / 64);
        const int64_t r0 = (int64_t)(blockIdx.x / kt) * 64, k0 = (int64_t)(blockIdx.x % kt) * 64;
        const int row = tid & 63, kq = tid >> 6;
        const T *src = A + min(r0 + row, m - 1);
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = src[min(k0 + kq + 4 * i, k - 1) * lda];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const bool in = r0 + row < m && k0 + kq + 4 * i < k;
            tile[row][kq + 4 * i] = in ? digit_rep(to_res<T>(x[i], mp), TOP, mp) : 0;
        }
        __syncthreads();
        const int orow = tid >> 2, ch = tid & 3;
        const size_t plane = (size_t)Mp * Kp;
        int8_t *dst = Al + (size_t)(r0 + orow) * Kp + k0 + ch * 16;
        union { int8_t b[16]; v4i v; } u[L];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            int32_t y = tile[orow][ch * 16 + e];
#pragma unroll
            for (int s = 0; s < L; ++s) u[s].b[e] = (int8_t)next_digit(y);
        }
#pragma unroll
        for (int s = 0; s < L; ++s) *reinterpret_cast<v4i *>(dst + s * plane) = u[s].v;
        return;
    }
    const int64_t quads = Kp / 4, total = Np * quads;
    const int64_t e0 = (int64_t)(blockIdx.x - na) * 1024 + tid;
    int64_t col[4], kk[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int64_t e = min(e0 + 256 * g, total - 1);
        col[g] = e / quads;
        kk[g] = (e % quads) * 4;
        const T *src = B + min(col[g], n - 1) * ldb;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[4 * g + i] = src[min(kk[g] + i, k - 1)];
    }
    const size_t plane = (size_t)Np * Kp;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t word[L];
#pragma unroll
        for (int s = 0; s < L; ++s) word[s] = 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = col[g] < n && kk[g] + i < k;
            int32_t y = in ? digit_rep(to_res<T>(x[4 * g + i], mp), TOP, mp) : 0;
#pragma unroll
            for (int s = 0; s < L; ++s) word[s] |= ((uint32_t)next_digit(y) & 255u) << (8 * i);
        }
        if (e0 + 256 * g < total) {
            int8_t *dst = Bl + (size_t)col[g] * Kp + kk[g];
#pragma unroll
            for (int s = 0; s < L; ++s) *reinterpret_cast<uint32_t *>(dst + s * plane) = word[s];
        }
    }
}

// Limb-form tile shapes: a BM x BN output tile per workgroup of WGM x WGN
// waves, each wave a (BM/WGM) x (BN/WGN) block of 32 x 32 blocks of
// v_mfma_i32_32x32x32_i8 (two k-steps per 64-deep stage), which sustains 1.4x
// or more of the int8 rate of the 16x16x64 form (4.36 vs 2.76 POP/s measured).
// LDS rows hold the 64 digits of one row (A) or column (B) for one K stage
// as four 16-byte chunks.  SWZ = 0: rows padded to 80 bytes.  SWZ = 1: rows of
// 64 bytes with chunk q of row r stored at slot q ^ ((r >> 2) & 3), so both
// the 16-lane row-wise fragment reads and the 4-lanes-per-row stores touch
// every bank group once.  DB = 1: two LDS stages; stage k+1 is stored while
// stage k feeds the MFMAs, with one barrier per stage.  DB = 2: in addition
// two register staging sets, so each global load has two stages to land.
template <int BM_, int BN_, int WGM_, int WGN_, int SWZ_ = 1, int DB_ = 0, int OCC_ = 1>
struct LimbShape {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, MF = 32, SWZ = SWZ_, DB = DB_;
    static constexpr int OCC = OCC_;  // waves per SIMD the register budget must allow
    static constexpr int NT = 64 * WGM * WGN;
    static constexpr int PITCH = SWZ ? 64 : 80;
};

typedef int v16i __attribute__((ext_vector_type(16)));

template <int SWZ> __device__ __forceinline__ int lds_slot(int row, int q)
{
    return SWZ ? (q ^ ((row >> 2) & 3)) : q;
}

template <int L, typename SH, typename TC, int EPI>
__global__ __launch_bounds__(SH::NT, SH::OCC) void k_gemm_limb(int64_t m, int64_t n, int64_t Kp,
                                                     const int8_t *__restrict__ Al, int64_t Mp,
                                                     const int8_t *__restrict__ Bl, int64_t Np,
                                                     TC *__restrict__ C, int64_t ldc, ModP mp, LimbW lw,
                                                     int64_t kslice, int64_t cslice,
                                                     const int *__restrict__ skip)
{
    if (skip && *skip) return;
    constexpr int BM = SH::BM, BN = SH::BN, NT = SH::NT, PITCH = SH::PITCH, SWZ = SH::SWZ;
    constexpr int NS = 2 * L - 1;
    constexpr int MF = SH::MF;
    constexpr int WM = BM / SH::WGM, WN = BN / SH::WGN;
    constexpr int FM = WM / MF, FN = WN / MF;
    constexpr int KS = 2;     // MFMA k-steps per 64-deep stage
    constexpr int AE = 16;    // accumulator elements per lane
    typedef v16i acc_t;
    constexpr int ACH = L * BM * (LBK / 16);  // 16-byte chunks of A per stage
    constexpr int BCH = L * BN * (LBK / 16);
    constexpr int NBUF = SH::DB ? 2 : 1;
    __shared__ __attribute__((aligned(16))) int8_t As[NBUF][L][BM][PITCH];
    __shared__ __attribute__((aligned(16))) int8_t Bs[NBUF][L][BN][PITCH];

    int64_t tm, tn;
    if (!tile_of_block(Mp / BM, Np / BN, &tm, &tn)) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave % SH::WGM, wn = wave / SH::WGM;
    const int64_t r0 = tm * BM;
    const int64_t c0 = tn * BN;
    const size_t aplane = (size_t)Mp * Kp, bplane = (size_t)Np * Kp;
    // K slice of this workgroup (whole K when kslice >= Kp)
    const int64_t kbeg = (int64_t)blockIdx.y * kslice;
    const int64_t kend = Kp - kbeg < kslice ? Kp : kbeg + kslice;
    C += blockIdx.y * cslice;

    acc_t acc[FM][FN][NS];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int u = 0; u < NS; ++u) acc[i][j][u] = acc_t{};

    constexpr int AR = (ACH + NT - 1) / NT, BR = (BCH + NT - 1) / NT;
    constexpr int NSET = SH::DB == 2 ? 2 : 1;
    v4i ra[NSET][AR], rb[NSET][BR];
    auto load = [&](int set, int64_t k0) {
#pragma unroll
        for (int i = 0; i < AR; ++i) {
            int idx = tid + NT * i;
            if (ACH % NT == 0 || idx < ACH) {
                int s = idx / (BM * 4), rem = idx % (BM * 4);
                int row = rem >> 2, ch = rem & 3;
                ra[set][i] = *reinterpret_cast<const v4i *>(Al + s * aplane + (size_t)(r0 + row) * Kp + k0 + ch * 16);
            }
        }
#pragma unroll
        for (int i = 0; i < BR; ++i) {
            int idx = tid + NT * i;
            if (BCH % NT == 0 || idx < BCH) {
                int s = idx / (BN * 4), rem = idx % (BN * 4);
                int col = rem >> 2, ch = rem & 3;
                rb[set][i] = *reinterpret_cast<const v4i *>(Bl + s * bplane + (size_t)(c0 + col) * Kp + k0 + ch * 16);
            }
        }
    };
    auto stash = [&](int set, int buf) {
#pragma unroll
        for (int i = 0; i < AR; ++i) {
            int idx = tid + NT * i;
            if (ACH % NT == 0 || idx < ACH) {
                int s = idx / (BM * 4), rem = idx % (BM * 4);
                int row = rem >> 2;
                *reinterpret_cast<v4i *>(&As[buf][s][row][lds_slot<SWZ>(row, rem & 3) * 16]) = ra[set][i];
            }
        }
#pragma unroll
        for (int i = 0; i < BR; ++i) {
            int idx = tid + NT * i;
            if (BCH % NT == 0 || idx < BCH) {
                int s = idx / (BN * 4), rem = idx % (BN * 4);
                int col = rem >> 2;
                *reinterpret_cast<v4i *>(&Bs[buf][s][col][lds_slot<SWZ>(col, rem & 3) * 16]) = rb[set][i];
            }
        }
    };
    // fragments: lane holds row (lane % MF) of the block and 16 digits of
    // k-chunk q = 2 ks + lane / 32
    v4i a[FM][KS][L], b[FN][KS][L];
    auto fragments = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int q = ks * 2 + (lane >> 5);
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int row = wm * WM + i * MF + (lane & (MF - 1));
#pragma unroll
                for (int s = 0; s < L; ++s)
                    a[i][ks][s] = *reinterpret_cast<const v4i *>(&As[buf][s][row][lds_slot<SWZ>(row, q) * 16]);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int col = wn * WN + j * MF + (lane & (MF - 1));
#pragma unroll
                for (int t = 0; t < L; ++t)
                    b[j][ks][t] = *reinterpret_cast<const v4i *>(&Bs[buf][t][col][lds_slot<SWZ>(col, q) * 16]);
            }
        }
    };
    auto mfmas = [&]() {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int s = 0; s < L; ++s)
#pragma unroll
                        for (int t = 0; t < L; ++t)
                            acc[i][j][s + t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[j][ks][t], a[i][ks][s],
                                                                                     acc[i][j][s + t], 0, 0, 0);
    };

    const int64_t nk = (kend - kbeg) / LBK;
    if constexpr (SH::DB == 2) {
        // stage kt lives in LDS buffer kt & 1; register set (kt + 1) & 1
        // holds stage kt + 1 and set kt & 1 receives stage kt + 2
        load(0, kbeg);
        if (nk > 1) load(1, kbeg + LBK);
        stash(0, 0);
        if (nk > 2) load(0, kbeg + 2 * LBK);
        __syncthreads();
        auto step = [&](int64_t kt, auto cur_c) {
            constexpr int cur = decltype(cur_c)::value;
            fragments(cur);
            if (kt + 1 < nk) stash(cur ^ 1, cur ^ 1);
            if (kt + 3 < nk) load(cur ^ 1, kbeg + (kt + 3) * LBK);
            mfmas();
            __syncthreads();
        };
        int64_t kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            step(kt, std::integral_constant<int, 0>());
            step(kt + 1, std::integral_constant<int, 1>());
        }
        if (kt < nk) step(kt, std::integral_constant<int, 0>());
    } else if constexpr (SH::DB == 1) {
        // stage kt lives in buffer kt & 1; the registers hold stage kt + 1
        load(0, kbeg);
        stash(0, 0);
        if (nk > 1) load(0, kbeg + LBK);
        __syncthreads();
        for (int64_t kt = 0; kt < nk; ++kt) {
            const int cur = (int)(kt & 1);
            fragments(cur);
            // buffer cur ^ 1 was last read before the previous barrier
            if (kt + 1 < nk) stash(0, cur ^ 1);
            if (kt + 2 < nk) load(0, kbeg + (kt + 2) * LBK);
            mfmas();
            __syncthreads();
        }
    } else {
        load(0, kbeg);
        for (int64_t kt = 0; kt < nk; ++kt) {
            stash(0, 0);
            __syncthreads();
            if (kt + 1 < nk) load(0, kbeg + (kt + 1) * LBK);
            fragments(0);
            mfmas();
            __syncthreads();
        }
    }

    // The blocks are computed transposed (B digits as the first operand), so
    // lane l holds row l % MF of C and a store instruction covers runs of MF
    // rows of a column: element e is column 8 (e / 4) + 4 (l / 32) + e % 4 of a
    // 32x32 block, 4 (l / 16) + e of a 16x16 one.  The old values of C, where
    // the epilogue needs them, are loaded together before the arithmetic (at
    // indices clamped into C).  4000 x 4000 -= K = 128, two digits, int32: 67
    // -> 34 us (one column run of 4 rows a lane, each digit sum reduced in
    // turn, loads between the stores); the memory traffic alone takes 26.
    const bool inside = r0 + BM <= m && c0 + BN <= n;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t gr = r0 + wm * WM + i * MF + (lane & (MF - 1));
            const int64_t gc = c0 + wn * WN + j * MF + 4 * (lane / MF);
            const bool row_ok = inside || gr < m;
            TC *const dst = C + (row_ok ? gr : 0);
            TC old[AE];
            if (EPI != EPI_STORE) {
#pragma unroll
                for (int e = 0; e < AE; ++e) {
                    const int64_t col = gc + 8 * (e >> 2) + (e & 3);
                    old[e] = dst[(inside ? col : min(col, n - 1)) * ldc];
                }
            }
#pragma unroll
            for (int e = 0; e < AE; ++e) {
                double tot;
                if (lw.lazy) {
                    tot = (double)acc[i][j][0][e];
#pragma unroll
                    for (int u = 1; u < NS; ++u) tot = fma((double)acc[i][j][u][e], lw.w[u], tot);
                } else {
                    const double d0 = (double)acc[i][j][0][e];
                    tot = fma(-rint(d0 * mp.pinv), mp.pd, d0);
#pragma unroll
                    for (int u = 1; u < NS; ++u) {
                        const double d = (double)acc[i][j][u][e];
                        tot = fma(fma(-rint(d * mp.pinv), mp.pd, d), lw.w[u], tot);
                    }
                }
                // |tot| < 2^53: the rounded quotient leaves a balanced residue
                tot = fma(-rint(tot * mp.pinv), mp.pd, tot);
                uint32_t r = (uint32_t)(tot < 0.0 ? tot + mp.pd : tot);
                if (EPI == EPI_SUB) r = submod(to_res<TC>(old[e], mp), r, mp);
                else if (EPI == EPI_ADD) r = addmod(to_res<TC>(old[e], mp), r, mp);
                const int64_t col = gc + 8 * (e >> 2) + (e & 3);
                if (inside || (row_ok && col < n)) dst[col * ldc] = from_res<TC>(r);
            }
        }
}

template <int L, typename SH, typename TC>
int limb_core(modp_ctx *ctx, const GemmArgs &g, int epi, const int8_t *Al, int64_t Mp, const int8_t *Bl, int64_t Np,
              int64_t Kp, const LimbW &lw, const Slices &sl)
{
    const dim3 grid(xcd_grid((Np / SH::BN) * (Mp / SH::BM)), (unsigned)sl.S);
    TimedLaunch tl(ctx, "gemm_limb");
    TC *C = (TC *)g.C;
    if (epi == EPI_STORE)
        k_gemm_limb<L, SH, TC, EPI_STORE><<<grid, SH::NT, 0, ctx->stream>>>(
            g.m, g.n, Kp, Al, Mp, Bl, Np, C, g.ldc, g.mp, lw, sl.kslice, sl.cslice, g.skip);
    else if (epi == EPI_SUB)
        k_gemm_limb<L, SH, TC, EPI_SUB><<<grid, SH::NT, 0, ctx->stream>>>(
            g.m, g.n, Kp, Al, Mp, Bl, Np, C, g.ldc, g.mp, lw, sl.kslice, sl.cslice, g.skip);
    else
        k_gemm_limb<L, SH, TC, EPI_ADD><<<grid, SH::NT, 0, ctx->stream>>>(
            g.m, g.n, Kp, Al, Mp, Bl, Np, C, g.ldc, g.mp, lw, sl.kslice, sl.cslice, g.skip);
    return hip_check(ctx, hipGetLastError(), "k_gemm_limb launch");
}

// tile_m x tile_n -> workgroup shape, all on 32x32 MFMA blocks with two
// register sets ahead of two LDS stages (measured on the planes alone).  Four
// digits on 64x64 hold seven weight planes of accumulators, which leave room
// for two waves on a SIMD only with one register set: 1500^3 64 us, with two
// sets and one wave 80; the trailing update 4000 x 4000 x 128 63 against 99.
//   64x64    2x2 waves; 1024^3, two digits 12.7 us (16x16 blocks, one stage:
//            14.6), 2501 x 1203 x 1777, three digits 58 (62.9), 5000^3 919 (1002)
//   128x64   two digits 2x2 waves, else 4x2; 3000^3, two digits 133 us (140;
//            64x64 136)
//   128x128  (one or two digits) one digit 2x2 waves, two 4x2
//   256x256  (one digit) 4x2 waves; 5000^3 177 us (128x128 tiles 219)
template <int L, typename TC>
int limb_by_shape(modp_ctx *ctx, const GemmArgs &g, int epi, const int8_t *Al, int64_t Mp, const int8_t *Bl,
                  int64_t Np, int64_t Kp, const LimbW &lw, int tile_m, int tile_n, const Slices &sl)
{
    if constexpr (L == 1)
        if (tile_m == 256)
            return limb_core<L, LimbShape<256, 256, 4, 2, 1, 2>, TC>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, sl);
    if constexpr (L <= 2)
        if (tile_m == 128 && tile_n == 128)
            return limb_core<L, LimbShape<128, 128, L == 1 ? 2 : 4, 2, 1, 2>, TC>(ctx, g, epi, Al, Mp, Bl, Np, Kp,
                                                                                     lw, sl);
    if (tile_m == 128 && tile_n == 64)
        return limb_core<L, LimbShape<128, 64, L == 2 ? 2 : 4, 2, 1, L == 4 ? 1 : 2>, TC>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw,
                                                                                sl);
    return limb_core<L, LimbShape<64, 64, 2, 2, 1, L == 4 ? 1 : 2, L == 4 ? 2 : 1>, TC>(ctx, g, epi, Al, Mp, Bl,
                                                                                           Np, Kp, lw, sl);
}

}  // namespace

template <int L>
int launch_limb_impl(modp_ctx *ctx, const GemmArgs &g, int epi, const int8_t *Al, int64_t Mp, const int8_t *Bl,
                     int64_t Np, int64_t Kp, const LimbW &lw, int tile_m, int tile_n, const Slices &sl)
{
    if (g.kc == EK_F64) return limb_by_shape<L, double>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tile_m, tile_n, sl);
    if (g.kc == EK_F32) return limb_by_shape<L, float>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tile_m, tile_n, sl);
    return limb_by_shape<L, int32_t>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tile_m, tile_n, sl);
}
