// gemm.hip -- mod-p GEMM cores for gfx950.
//
// Plain form: FP64 MFMA (v_mfma_f64_16x16x4f64) on balanced residues of
// magnitude at most (p+1)/2, with the accumulators reduced every R k4-steps
// so that every partial sum stays an exact integer below 2^53 (the
// reference's stripe bound, src/CuModMatrix/kernel_mul/stripe_mul.jl:13-27,
// applied per MFMA step instead of per cuBLAS stripe).
//
// Limb form (kernels in gemm_limb.h): residues as signed base-256 digits in
// int8 on v_mfma_i32_32x32x32_i8; this file splits the operands into digit
// planes, cuts K into int32-safe chunks and picks the launch.
//
// Both forms can cut K into slices that run concurrently (blockIdx.y) and are
// summed mod p afterwards, for products whose output grid alone leaves CUs
// idle.
#include <algorithm>

#include "gemm_limb.h"
#include "gemm_tile.h"

namespace {

// --------------------------------------------------------------------------
// plain FP64 form
// --------------------------------------------------------------------------

// blockIdx.y selects a K slice [y*kslice, (y+1)*kslice); slice y writes its
// residues at C + y*cslice (one slice: kslice >= k, cslice = 0).
template <typename TA, typename TB, typename TC, int BM, int BN, int EPI, int RED>
__global__ __launch_bounds__(256, 2) void k_gemm_f64(int64_t m, int64_t n, int64_t k,
                                                  const TA *__restrict__ A, int64_t lda,
                                                  const TB *__restrict__ B, int64_t ldb,
                                                  TC *__restrict__ C, int64_t ldc, ModP mp, int rq,
                                                  int64_t kslice, int64_t cslice,
                                                  const int *__restrict__ skip)
{
    if (skip && *skip) return;
    int64_t tm, tn;
    if (!tile_of_block((m + BM - 1) / BM, (n + BN - 1) / BN, &tm, &tn)) return;
    const int64_t kb = (int64_t)blockIdx.y * kslice;
    const int64_t klen = k - kb < kslice ? k - kb : kslice;
    __shared__ F64Smem<BM, BN> sm;
    gemm_f64_tile<TA, TB, TC, BM, BN, EPI, RED>(m, n, klen, A + kb * lda, lda, B + kb, ldb, C + blockIdx.y * cslice,
                                                ldc, mp, rq, tm * BM, tn * BN, sm);
}

// The plain form of a small product: one workgroup per 16 x 16 block of C,
// its four waves taking a quarter of K each and their residues summed in LDS.
// Such a product is bound by latency, so there are no LDS stages and no
// barriers before the sum: a wave loads the MFMA fragments of eight k4-steps
// straight from the operands (16 runs of 16 rows of A, 16 columns of B), all
// before it uses one.  The block is computed transposed, so a lane holds one
// row.  48 x 40 x 56 mod 11: 8.6 -> 3.5 us (64 x 64 tiles in stages of 16 k).
// blockIdx.y: products at the strides sa, sb and sc, the last of its own size.
template <typename T, typename TC, int EPI>
__global__ __launch_bounds__(256) void k_gemm_f64_small(int64_t m, int64_t n, int64_t k, const T *__restrict__ A,
                                                        int64_t lda, const T *__restrict__ B, int64_t ldb,
                                                        TC *__restrict__ C, int64_t ldc, ModP mp, int R,
                                                        int64_t sa, int64_t sb, int64_t sc, GemmSize last,
                                                        const int *__restrict__ skip)
{
    if (skip && *skip) return;
    A += blockIdx.y * sa;
    B += blockIdx.y * sb;
    C += blockIdx.y * sc;
    if (blockIdx.y + 1 == gridDim.y) {
        m = last.m;
        n = last.n;
        k = last.k;
    }
    constexpr int U = 8;
    __shared__ double part[4][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t mt = (m + 15) / 16;
    const int64_t r0 = (blockIdx.x % mt) * 16, c0 = (blockIdx.x / mt) * 16;
    if (c0 >= n) return;
    const int64_t kq = (k + 15) / 16 * 4;  // a wave's share of K, in whole k4-steps
    const int64_t kbeg = wave * kq, kend = min(k, kbeg + kq);
    const int64_t row = r0 + (lane & 15), col = c0 + (lane & 15);
    const bool row_ok = row < m, col_ok = col < n;
    const T *a = A + (row_ok ? row : 0), *b = B + (col_ok ? col : 0) * ldb;
    const int q = lane >> 4;
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    int cnt = 0;
    for (int64_t k0 = kbeg; k0 < kend; k0 += 4 * U) {
        T xa[U], xb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t kk = min(k0 + 4 * u + q, k - 1);
            xa[u] = a[kk * lda];
            xb[u] = b[kk];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = k0 + 4 * u + q < kend;
            const double fa = in && row_ok ? bal_of<T>(xa[u], mp) : 0.0;
            const double fb = in && col_ok ? bal_of<T>(xb[u], mp) : 0.0;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(fb, fa, acc, 0, 0, 0);
            if (++cnt == R) {
                cnt = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fma(-rint(acc[e] * mp.pinv), mp.pd, acc[e]);
            }
        }
    }
    // lane: row lane % 16, columns lane / 16 + 4 e
#pragma unroll
    for (int e = 0; e < 4; ++e)
        part[wave][q + 4 * e][lane & 15] = fma(-rint(acc[e] * mp.pinv), mp.pd, acc[e]);
    __syncthreads();
    const int rl = tid & 15, cl = tid >> 4;
    const double s = part[0][cl][rl] + part[1][cl][rl] + part[2][cl][rl] + part[3][cl][rl];
    if (r0 + rl < m && c0 + cl < n) {
        uint32_t v = (uint32_t)dmod(s, mp);
        TC *dst = C + (r0 + rl) + (c0 + cl) * ldc;
        if (EPI == EPI_SUB) v = submod(to_res<TC>(*dst, mp), v, mp);
        *dst = from_res<TC>(v);
    }
}

// C = epi(C, sum of S slice results mod p); slice s holds m x n residues at
// P + s*m*n (leading dimension m).
template <typename TC, int EPI>
__global__ __launch_bounds__(256) void k_slice_sum(int64_t m, int64_t n, const int32_t *__restrict__ P, int S,
                                                   TC *__restrict__ C, int64_t ldc, ModP mp,
                                                   const int *__restrict__ skip)
{
    if (skip && *skip) return;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t mn = m * n;
    if (idx >= mn) return;
    double acc = 0.0;  // S * p < 2^53
    for (int s = 0; s < S; ++s) acc += (double)P[(int64_t)s * mn + idx];
    uint32_t r = (uint32_t)dmod(acc, mp);
    TC *dst = C + idx % m + (idx / m) * ldc;
    if (EPI == EPI_SUB) r = submod(to_res<TC>(*dst, mp), r, mp);
    else if (EPI == EPI_ADD) r = addmod(to_res<TC>(*dst, mp), r, mp);
    *dst = from_res<TC>(r);
}

// y = A x mod p (A m x k column-major, x and y contiguous), bound by reading A
// once.  A wave reads 16 bytes a lane, 1 KiB of a column, and keeps sixteen such
// loads in flight; the four waves of a workgroup take quarters of its K slice
// (blockIdx.y) and meet in LDS.  Elements are balanced by one rounded quotient
// (at most h = (p + 1) / 2 + 2 in magnitude) and the FP64 sum is reduced every
// `cadence` columns, so that it stays exact.  Several slices leave their residues in P
// and the last one of a row block to arrive sums them (stores and loads at
// agent scope, since the slices run on all XCDs); it also resets the count.
// 6001 x 7003 in FP64: 64 us, 5.3 TB/s (one row a lane and the slices' sum in
// a launch of its own: 89); 1000 x 1000 9 us (44).
constexpr int GV_U = 8;  // columns of a batch
template <typename T, int V> struct __attribute__((packed, aligned(sizeof(T)))) RowsOf {
    T v[V];
};
template <typename T, int V>
__global__ __launch_bounds__(256) void k_gemv(int64_t m, int64_t k, const T *__restrict__ A, int64_t lda,
                                              const T *__restrict__ x, T *__restrict__ y, int32_t *__restrict__ P,
                                              int *__restrict__ arrived, int64_t kslice, int cadence, ModP mp)
{
    __shared__ double s_acc[4][64 * V];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t r = (int64_t)blockIdx.x * (64 * V) + lane * V;
    const int64_t rb = min(r, m - V);  // (m >= V) the last lanes read again what they share
    const int64_t c0 = (int64_t)blockIdx.y * kslice + wave * (kslice / 4);
    const int64_t c1 = min(k, c0 + kslice / 4);
    double acc[V];
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = 0.0;
    auto reduce = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = fma(-rint(acc[e] * mp.pinv), mp.pd, acc[e]);
    };
    if (c0 < c1) {
        const int nb = (int)((c1 - c0 + GV_U - 1) / GV_U);
        RowsOf<T, V> a[2][GV_U];
        auto load = [&](int i, RowsOf<T, V> *d) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < GV_U; ++q)
                d[q] = *(const RowsOf<T, V> *)(A + rb + min(c0 + (int64_t)i * GV_U + q, c1 - 1) * lda);
        };
        // 64 elements of x, one a lane; zero past the end
        auto load_x = [&](int64_t c) __attribute__((always_inline)) {
            const T v = x[min(c + lane, c1 - 1)];
            return c + lane < c1 ? bal_of<T>(v, mp) : 0.0;
        };
        load(0, a[0]);
        double xv = load_x(c0);
        int since = 0;
        auto batch = [&](int i, const RowsOf<T, V> *d) __attribute__((always_inline)) {
            const int at = (i * GV_U) & 63;
#pragma unroll
            for (int q = 0; q < GV_U; ++q) {
                const uint64_t b = __builtin_bit_cast(uint64_t, xv);
                const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, at + q);
                const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), at + q);
                const double xq = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
#pragma unroll
                for (int e = 0; e < V; ++e) acc[e] = fma(bal_of<T>(d[q].v[e], mp), xq, acc[e]);
                if (q == 3 && cadence == 4) reduce();
            }
            since += GV_U;
            if (since >= cadence) {
                reduce();
                since = 0;
            }
        };
        for (int i = 0; i < nb; i += 2) {
            load(i + 1, a[1]);
            if (i != 0 && ((i * GV_U) & 63) == 0) xv = load_x(c0 + (int64_t)i * GV_U);
            batch(i, a[0]);
            if (i + 1 < nb) {
                load(i + 2, a[0]);
                batch(i + 1, a[1]);
            }
        }
        reduce();
    }
#pragma unroll
    for (int e = 0; e < V; ++e)
        if (rb + e >= r) s_acc[wave][(int)(rb - (r - lane * V)) + e] = acc[e];
    __syncthreads();
    const int64_t row = (int64_t)blockIdx.x * (64 * V) + tid;
    const bool mine = tid < 64 * V && row < m;
    uint32_t v = 0;
    if (mine) v = (uint32_t)dmod((s_acc[0][tid] + s_acc[1][tid]) + (s_acc[2][tid] + s_acc[3][tid]), mp);
    if (!P) {
        if (mine) y[row] = from_res<T>(v);
        return;
    }
    if (mine)
        __hip_atomic_store(P + (int64_t)blockIdx.y * m + row, (int32_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!arrived) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
        const int S = (int)gridDim.y;
        s_last = atomicAdd(arrived + blockIdx.x, 1) == S - 1;
        if (s_last) __hip_atomic_store(arrived + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    // the threads of a row take every G-th slice each
    constexpr int R = 64 * V, G = 256 / R, U = 16;
    const int S = (int)gridDim.y;
    const int64_t row2 = (int64_t)blockIdx.x * R + tid % R;
    double sum = 0.0;  // fewer than 2^26 slices
    for (int t = tid / R; t < S; t += G * U) {
        int32_t w[U];
#pragma unroll
        for (int q = 0; q < U; ++q)
            w[q] = __hip_atomic_load(P + (int64_t)min(t + G * q, S - 1) * m + min(row2, m - 1), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int q = 0; q < U; ++q) sum += t + G * q < S ? (double)w[q] : 0.0;
    }
    s_acc[tid / R][tid % R] = sum;
    __syncthreads();
    if (!mine) return;
    sum = 0.0;
#pragma unroll
    for (int q = 0; q < G; ++q) sum += s_acc[q][tid];
    y[row] = from_res<T>((uint32_t)dmod(sum, mp));
}

__global__ void k_zero_ints(int *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

int64_t round_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

// whether the address ranges [a0, a1) and [b0, b1) have a byte in common
bool meet(const void *a0, const void *a1, const void *b0, const void *b1)
{
    return (const char *)a0 < (const char *)b1 && (const char *)b0 < (const char *)a1;
}

// whether C lies (partly) in the memory of A or B
bool over_operand(const GemmArgs &g)
{
    auto bytes = [](int kind) -> int64_t { return kind == EK_F64 ? 8 : 4; };
    auto end = [&](const void *X, int64_t rows, int64_t cols, int64_t ld, int kind) {
        return (const char *)X + ((cols - 1) * ld + rows) * bytes(kind);
    };
    if (g.m <= 0 || g.n <= 0 || g.k <= 0) return false;
    const char *const c1 = end(g.C, g.m, g.n, g.ldc, g.kc);
    return meet(g.C, c1, g.A, end(g.A, g.m, g.k, g.lda, g.ka)) || meet(g.C, c1, g.B, end(g.B, g.k, g.n, g.ldb, g.kb));
}

// ---- dispatch helpers -----------------------------------------------------

template <typename TA, typename TB, typename TC, int BM, int BN, int EPI>
int launch_f64_e(modp_ctx *ctx, const GemmArgs &g, int R, const Slices &sl, const dim3 &grid)
{
    const TA *A = (const TA *)g.A;
    const TB *B = (const TB *)g.B;
    TC *C = (TC *)g.C;
    int rq = 1;
    const int red = f64_reduce_mode(R, sl.kslice < g.k ? sl.kslice : g.k, &rq);
#define F64_LAUNCH(RED_)                                                                                      \
    k_gemm_f64<TA, TB, TC, BM, BN, EPI, RED_><<<grid, 256, 0, ctx->stream>>>(g.m, g.n, g.k, A, g.lda, B, g.ldb, C, \
                                                                            g.ldc, g.mp, rq, sl.kslice,          \
                                                                            sl.cslice, g.skip)
    switch (red) {
    case RED_NONE: F64_LAUNCH(RED_NONE); break;
    case RED_STAGE: F64_LAUNCH(RED_STAGE); break;
    case RED_2: F64_LAUNCH(RED_2); break;
    default: F64_LAUNCH(RED_STEP); break;
    }
#undef F64_LAUNCH
    return hip_check(ctx, hipGetLastError(), "k_gemm_f64 launch");
}

template <typename TA, typename TC, int EPI>
int launch_f64_tile(modp_ctx *ctx, const GemmArgs &g, int R, int tile, const Slices &sl)
{
    TimedLaunch tl(ctx, "gemm_f64");
    if (tile == 128) {
        const dim3 grid(xcd_grid(((g.n + 127) / 128) * ((g.m + 127) / 128)), (unsigned)sl.S);
        return launch_f64_e<TA, TA, TC, 128, 128, EPI>(ctx, g, R, sl, grid);
    }
    const dim3 grid(xcd_grid(((g.n + 63) / 64) * ((g.m + 63) / 64)), (unsigned)sl.S);
    return launch_f64_e<TA, TA, TC, 64, 64, EPI>(ctx, g, R, sl, grid);
}

// The operand / result / epilogue combinations the library uses: user
// products (C of the operands' type, or int32 K-slice partials), and the
// int32 working arrays of elimination and inversion (subtracting updates,
// products into the caller's storage type).
int launch_f64(modp_ctx *ctx, const GemmArgs &g, int R, int tile, const Slices &sl)
{
    if (g.ka == g.kb) {
        if (g.epi == EPI_STORE) {
            if (g.ka == EK_F64 && g.kc == EK_F64) return launch_f64_tile<double, double, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_F64 && g.kc == EK_I32) return launch_f64_tile<double, int32_t, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_F32 && g.kc == EK_F32) return launch_f64_tile<float, float, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_F32 && g.kc == EK_I32) return launch_f64_tile<float, int32_t, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_I32 && g.kc == EK_I32) return launch_f64_tile<int32_t, int32_t, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_I32 && g.kc == EK_F64) return launch_f64_tile<int32_t, double, EPI_STORE>(ctx, g, R, tile, sl);
            if (g.ka == EK_I32 && g.kc == EK_F32) return launch_f64_tile<int32_t, float, EPI_STORE>(ctx, g, R, tile, sl);
        } else if (g.epi == EPI_SUB && g.ka == EK_I32 && g.kc == EK_I32) {
            return launch_f64_tile<int32_t, int32_t, EPI_SUB>(ctx, g, R, tile, sl);
        }
    }
    return set_error(ctx, MODP_ERR_DTYPE, "FP64 GEMM: unsupported operand combination (%d, %d, %d, epilogue %d)",
                     g.ka, g.kb, g.kc, g.epi);
}

// Blocks of 16 x 16 times K, what k_gemm_f64_small reads (every block its own
// rows and columns), if it takes the product at all: at most 1024 blocks (four
// workgroups per CU; 1024^2 x 32, 4096 blocks: 21 us against 7.8 in 64 x 64
// tiles) and K up to 1024; else -1.
int64_t small_work(int64_t m, int64_t n, int64_t k)
{
    const int64_t blocks = ((m + 15) / 16) * ((n + 15) / 16);
    return blocks <= 1024 && k <= 1024 && k > 0 ? blocks * k : -1;
}
// against 64 x 64 tiles it pays up to 512 x 512 x 256 (11.9 us, 23 in tiles), but
// not while those take one stage of K, or two in a single tile: 6.0 us from 64 x 64
// to 512 x 512 at k = 16, where this takes 6.5 to 7.3 (one call after the other)
bool f64_small(const GemmArgs &g)
{
    const int64_t w = small_work(g.m, g.n, g.k);
    const bool short_k = g.k <= PBK || (g.k <= 2 * PBK && g.m <= 64 && g.n <= 64);
    return w >= 0 && w <= 262144 && !short_k && g.ka == g.kb && g.ka == g.kc &&
           (g.epi == EPI_STORE || (g.epi == EPI_SUB && g.kc == EK_I32));
}
int launch_f64_small(modp_ctx *ctx, const GemmArgs &g, int R, int64_t count, int64_t sa, int64_t sb, int64_t sc,
                     const GemmSize &last)
{
    TimedLaunch tl(ctx, "gemm_f64_small");
    const unsigned grid = (unsigned)(((g.m + 15) / 16) * ((g.n + 15) / 16));
#define SMALL(T_, EPI_)                                                                                             \
    k_gemm_f64_small<T_, T_, EPI_><<<dim3(grid, (unsigned)count), 256, 0, ctx->stream>>>(g.m, g.n, g.k, (const T_ *)g.A, g.lda,             \
                                                                  (const T_ *)g.B, g.ldb, (T_ *)g.C, g.ldc, g.mp, R, \
                                                                  sa, sb, sc, last, g.skip)
    if (g.ka == EK_F64) SMALL(double, EPI_STORE);
    else if (g.ka == EK_F32) SMALL(float, EPI_STORE);
    else if (g.epi == EPI_STORE) SMALL(int32_t, EPI_STORE);
    else SMALL(int32_t, EPI_SUB);
#undef SMALL
    return hip_check(ctx, hipGetLastError(), "k_gemm_f64_small launch");
}

template <typename TC>
int launch_slice_sum_t(modp_ctx *ctx, const GemmArgs &g, int epi, const int32_t *P, int S)
{
    const int64_t mn = g.m * g.n;
    const unsigned grid = (unsigned)((mn + 255) / 256);
    TC *C = (TC *)g.C;
    if (epi == EPI_STORE)
        k_slice_sum<TC, EPI_STORE><<<grid, 256, 0, ctx->stream>>>(g.m, g.n, P, S, C, g.ldc, g.mp, g.skip);
    else if (epi == EPI_SUB)
        k_slice_sum<TC, EPI_SUB><<<grid, 256, 0, ctx->stream>>>(g.m, g.n, P, S, C, g.ldc, g.mp, g.skip);
    else
        k_slice_sum<TC, EPI_ADD><<<grid, 256, 0, ctx->stream>>>(g.m, g.n, P, S, C, g.ldc, g.mp, g.skip);
    return hip_check(ctx, hipGetLastError(), "k_slice_sum launch");
}

int launch_slice_sum(modp_ctx *ctx, const GemmArgs &g, int epi, const int32_t *P, int S)
{
    if (g.kc == EK_F64) return launch_slice_sum_t<double>(ctx, g, epi, P, S);
    if (g.kc == EK_F32) return launch_slice_sum_t<float>(ctx, g, epi, P, S);
    return launch_slice_sum_t<int32_t>(ctx, g, epi, P, S);
}

// slice results go to a workspace of S * m * n int32 residues
int32_t *slice_buffer(modp_ctx *ctx, const GemmArgs &g, int S, int *st)
{
    return (int32_t *)ws_get(ctx, WS_SLICES, sizeof(int32_t) * (size_t)S * (size_t)g.m * (size_t)g.n, st);
}

// digit planes of k in [kbeg, kbeg + kc) of both operands (of one type)
template <typename T>
int split_t(modp_ctx *ctx, const GemmArgs &g, int64_t kbeg, int64_t kc, int8_t *Al, int64_t Mp, int8_t *Bl, int64_t Np,
            int64_t Kp, int L)
{
    const unsigned na = (unsigned)((Mp / 64) * (Kp / 64));
    const unsigned nb = (unsigned)((Np * (Kp / 4) + 1023) / 1024);
    const T *A = (const T *)g.A + kbeg * g.lda, *B = (const T *)g.B + kbeg;
    TimedLaunch tl(ctx, "gemm_split");
#define SPLIT(L_)                                                                                                  \
    k_split_ab<T, L_><<<na + nb, 256, 0, ctx->stream>>>(g.m, g.n, kc, A, g.lda, B, g.ldb, Al, Mp, Bl, Np, Kp, na, \
                                                        g.mp, g.skip)
    switch (L) {
    case 1: SPLIT(1); break;
    case 2: SPLIT(2); break;
    case 3: SPLIT(3); break;
    default: SPLIT(4); break;
    }
#undef SPLIT
    return hip_check(ctx, hipGetLastError(), "k_split_ab launch");
}

int launch_limb(modp_ctx *ctx, const GemmArgs &g, int L, int epi, const int8_t *Al, int64_t Mp,
                const int8_t *Bl, int64_t Np, int64_t Kp, const LimbW &lw, int tm, int tn, const Slices &sl)
{
    switch (L) {
    case 1: return launch_limb_impl<1>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl);
    case 2: return launch_limb_impl<2>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl);
    case 3: return launch_limb_impl<3>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl);
    default: return launch_limb_impl<4>(ctx, g, epi, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl);
    }
}

int64_t tiles_of(const GemmArgs &g, int tm, int tn) { return ((g.m + tm - 1) / tm) * ((g.n + tn - 1) / tn); }

// slices of a K extent: S0 requested, each a multiple of `align` and at
// least `minlen` long
Slices make_slices(int64_t kext, int S0, int64_t align, int64_t minlen)
{
    Slices sl;
    if (S0 <= 1 || kext <= minlen) {
        sl.S = 1;
        sl.kslice = kext > 0 ? kext : 1;
        return sl;
    }
    int64_t ks = round_up((kext + S0 - 1) / S0, align);
    if (ks < minlen) ks = round_up(minlen, align);
    sl.S = (int)((kext + ks - 1) / ks);
    sl.kslice = ks;
    return sl;
}

int gemm_plain_cfg(modp_ctx *ctx, const GemmArgs &g, const GemmConfig &cfg)
{
    if (g.m <= 0 || g.n <= 0) return MODP_OK;
    const int R = f64_reduce_interval(g.mp.p);
    if (R < 1) return set_error(ctx, MODP_ERR_MODULUS_RANGE, "modulus %lld too large for the FP64 form", (long long)g.mp.p);
    // a C over an operand is written only after all workgroups have read it:
    // through the residues of the slices, also where there is one slice (a
    // single tile's workgroup has read everything before it stores)
    const bool over = over_operand(g);
    if (!over && f64_small(g)) return launch_f64_small(ctx, g, R, 1, 0, 0, 0, GemmSize{g.m, g.n, g.k});
    const int tile = cfg.tile_m == 128 ? 128 : 64;
    Slices sl = make_slices(g.k, cfg.ksplit, PBK, 64);
    if (sl.S == 1) {
        sl.kslice = g.k > 0 ? g.k : 1;
        if (!over || (g.m <= 64 && g.n <= 64)) return launch_f64(ctx, g, R, tile, sl);
    }
    int st = MODP_OK;
    int32_t *P = slice_buffer(ctx, g, sl.S, &st);
    if (!P) return st;
    GemmArgs gs = g;
    gs.C = P; gs.ldc = g.m; gs.kc = EK_I32; gs.epi = EPI_STORE;
    sl.cslice = g.m * g.n;
    MODP_TRY(launch_f64(ctx, gs, R, tile, sl));
    return launch_slice_sum(ctx, g, g.epi, P, sl.S);
}

// Output tile that a limb configuration's workgroups take.  With one digit
// the 128x128 configuration runs 256x256 tiles (twice the MFMA work per LDS
// byte) on products with at least one for every two CUs and a K that pays for
// their longer epilogue: float32 mod 127, 3072^3 73.6 us against 80.9, 4096^3
// 115 against 131, 5000^3 222 against 263, 8192^3 743 against 928; but 2560^3
// (100 tiles) 63.5 against 49.3, 3000 x 6000 x 500 55.9 against 43.6.
void limb_tile(const GemmConfig &cfg, int L, int64_t m, int64_t n, int64_t k, bool wide, int *tm, int *tn)
{
    *tm = cfg.tile_m >= 128 ? 128 : 64;
    *tn = (*tm == 128 && cfg.tile_n >= 128 && L <= 2) ? 128 : 64;
    if (wide && L == 1 && *tn == 128 && k >= 1536 && ((m + 255) / 256) * ((n + 255) / 256) >= 128) *tm = *tn = 256;
}

// ext: caller-provided workspace for the digit planes (no allocation); the
// planes of each K chunk must fit in ext->bytes and the launch has one K slice
int gemm_limb_cfg(modp_ctx *ctx, const GemmArgs &g, const GemmConfig &cfg, const LimbScratch *ext = nullptr)
{
    if (g.m <= 0 || g.n <= 0) return MODP_OK;
    const int L = limb_count(g.mp.p);
    if (L > 4) return set_error(ctx, MODP_ERR_MODULUS_RANGE, "modulus %lld needs more than 4 limbs", (long long)g.mp.p);
    // largest k-chunk whose shift sums fit int32: a digit product is at most
    // 128^2 in magnitude and shift L-1 collects L of them per k, so
    // L * K * 2^14 <= 2^31 - 1
    const int64_t pairs = L;
    int64_t kmax = ((int64_t)2147483647 / (pairs * 16384)) / LBK * LBK;
    int tm, tn;
    limb_tile(cfg, L, g.m, g.n, g.k, !ext, &tm, &tn);
    const int64_t Mp = round_up(g.m, tm), Np = round_up(g.n, tn);
    LimbW lw;
    {
        double w = 1.0;
        for (int u = 0; u < 7; ++u) {
            lw.w[u] = w > (double)g.mp.half ? w - g.mp.pd : w;
            w = fmod(w * 256.0, (double)g.mp.p);
        }
    }
    lw.lazy = limb_lazy(L, g.k < kmax ? g.k : kmax, g.mp.p);
    if (g.ka != g.kb)
        return set_error(ctx, MODP_ERR_DTYPE, "digit form: operands of different types (%d, %d)", g.ka, g.kb);
    if (g.k <= 0)  // C unchanged, or zero
        return g.epi != EPI_STORE ? MODP_OK
                                  : hip_check(ctx, hipMemset2DAsync(g.C, (size_t)g.ldc * (g.kc == EK_F64 ? 8 : 4), 0,
                                                                    (size_t)g.m * (g.kc == EK_F64 ? 8 : 4),
                                                                    (size_t)g.n, ctx->stream), "hipMemset2DAsync");
    int64_t kdone = 0;
    bool first = true;
    do {
        int64_t kc = g.k - kdone;
        if (kc > kmax) kc = kmax;
        const int64_t Kp = round_up(kc, LBK);
        int st = MODP_OK;
        int8_t *Al, *Bl;
        if (ext) {
            const size_t need = (size_t)L * (size_t)(Mp + Np) * (size_t)Kp;
            if (need > ext->bytes || cfg.ksplit != 1)
                return set_error(ctx, MODP_ERR_ARG, "digit planes of %zu bytes exceed the %zu-byte workspace", need,
                                 ext->bytes);
            Al = ext->base;
            Bl = ext->base + (size_t)L * Mp * Kp;
        } else {
            Al = (int8_t *)ws_get(ctx, WS_ALIMB, (size_t)L * Mp * Kp, &st);
            if (!Al) return st;
            Bl = (int8_t *)ws_get(ctx, WS_BLIMB, (size_t)L * Np * Kp, &st);
            if (!Bl) return st;
        }
        if (g.ka == EK_F64) MODP_TRY(split_t<double>(ctx, g, kdone, kc, Al, Mp, Bl, Np, Kp, L));
        else if (g.ka == EK_F32) MODP_TRY(split_t<float>(ctx, g, kdone, kc, Al, Mp, Bl, Np, Kp, L));
        else MODP_TRY(split_t<int32_t>(ctx, g, kdone, kc, Al, Mp, Bl, Np, Kp, L));
        int epi = g.epi;
        if (!first && epi == EPI_STORE) epi = EPI_ADD;
        Slices sl = make_slices(Kp, cfg.ksplit, LBK, 256);
        if (sl.S == 1) {
            sl.kslice = Kp;
            MODP_TRY(launch_limb(ctx, g, L, epi, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl));
        } else {
            int32_t *P = slice_buffer(ctx, g, sl.S, &st);
            if (!P) return st;
            GemmArgs gs = g;
            gs.C = P; gs.ldc = g.m; gs.kc = EK_I32;
            sl.cslice = g.m * g.n;
            MODP_TRY(launch_limb(ctx, gs, L, EPI_STORE, Al, Mp, Bl, Np, Kp, lw, tm, tn, sl));
            MODP_TRY(launch_slice_sum(ctx, g, epi, P, sl.S));
        }
        kdone += kc;
        first = false;
    } while (kdone < g.k);
    return MODP_OK;
}

}  // namespace

int limb_count(int64_t p)
{
    // signed base-256 digits: L digits represent every residue class iff p <= 256^L
    int L = 1;
    while (L < 8 && p > ((int64_t)1 << (8 * L))) ++L;
    return L;
}

int choose_form(int64_t m, int64_t n, int64_t k, int64_t p)
{
    // small products: one launch of the plain form's small kernel against the
    // digit form's two, up to 512 x 512 x 128 (7.4 us against 10.0 to 12.7)
    const int64_t w = small_work(m, n, k);
    if (w >= 0 && w <= 131072) return MODP_FORM_PLAIN_F64;
    // shallow ones: the digit form's split passes and its epilogue against the
    // plain form's k-steps.  2048^2: at k = 32 13.3, 15.2 and 26 us with one,
    // two and four digits against 15.8, at k = 64 13.4, 15.4 and 26 against 22,
    // at k = 128 13.8, 16.5 and 28 against 34.  Up to about 1000 x 1000 the digit
    // form's second launch weighs more (1000^2 at k = 48 9.6, 10.4 and 10.8 us with
    // one, two and three digits against 8.9, at k = 72 9.8, 11.0 and 12.0 against
    // 11.2), and so do the planes of a long thin product while the plain form takes
    // 64x64 tiles there (64 x 40,000 at k = 48 14.1, 16.4, 20.6 and 24.3 against
    // 15.5 to 17, at k = 96 17.3, 20.2, 24.9 and 29.1 against 22.7 to 25.8)
    static const int wide[4] = {48, 48, 56, 96}, few[4] = {56, 64, 88, 96}, thin[4] = {48, 56, 112, 112};
    auto tiles = [&](int64_t t) { return ((m + t - 1) / t) * ((n + t - 1) / t); };
    const int *from = std::min(m, n) <= 64 && tiles(64) > 256 && tiles(128) < 512 ? thin : m * n <= 1 << 20 ? few : wide;
    return k >= from[std::min(limb_count(p), 4) - 1] ? MODP_FORM_LIMB_I8 : MODP_FORM_PLAIN_F64;
}

bool gemm_config_valid(const GemmArgs &g, const GemmConfig &cfg)
{
    if (cfg.ksplit < 1 || cfg.ksplit > 16) return false;
    const bool sq64 = cfg.tile_m == 64 && cfg.tile_n == 64;
    const bool sq128 = cfg.tile_m == 128 && cfg.tile_n == 128;
    const bool r128x64 = cfg.tile_m == 128 && cfg.tile_n == 64;
    if (cfg.form == MODP_FORM_PLAIN_F64) return (sq64 || sq128) && f64_reduce_interval(g.mp.p) >= 1;
    if (cfg.form == MODP_FORM_RNS_I8) {
        const bool sq256 = cfg.tile_m == 256 && cfg.tile_n == 256;
        return (sq128 || sq256) && cfg.ksplit == 1 && rns_planes(g.mp.p, g.k < RNS_KCHUNK ? g.k : RNS_KCHUNK) > 0;
    }
    // 128x128 limb tiles hold 2L-1 accumulators of a 64x64 block per wave:
    // register room for L <= 2 only
    if (cfg.form == MODP_FORM_LIMB_I8) {
        const int L = limb_count(g.mp.p);
        return (sq64 || r128x64 || (sq128 && L <= 2)) && L <= 4;
    }
    return false;
}

// The RNS form's r moduli against the limb form's L^2 digit products: it pays
// when it issues at most three quarters of the limb form's MFMA work and the
// product is large enough for its two more launches and its residue planes of
// C.  Four digits: 2501 x 1203 x 1777 121 us against 111, 2048^3 126 against
// 159.  One plane (p <= 255) issues what one digit does (mod 127, one plane
// against one digit: float64 6000^3 495 us and 450, 8192^3 920 and 860, 10,000^3
// 1550 and 1610, 12,000^3 2390 and 2380; float32 8192^3 845 and 750).  From four
// 256 x 256 output tiles per CU it is what modp_gemm_config_get has always
// answered, and stays.
static bool rns_pays(const modp_ctx *ctx, const GemmArgs &g)
{
    const int L = limb_count(g.mp.p);
    const int r = rns_planes(g.mp.p, g.k < RNS_KCHUNK ? g.k : RNS_KCHUNK);
    if (r == 1) return tiles_of(g, 256, 256) >= 4 * ctx->num_cus;
    return r > 0 && 4 * r <= 3 * L * L && (double)g.m * (double)g.n * (double)g.k >= 6.5e9;
}

GemmConfig gemm_default_config(const modp_ctx *ctx, const GemmArgs &g, int form)
{
    GemmConfig c;
    c.form = form == MODP_FORM_AUTO ? choose_form(g.m, g.n, g.k, g.mp.p) : form;
    if (form == MODP_FORM_AUTO && c.form == MODP_FORM_LIMB_I8 && rns_pays(ctx, g)) c.form = MODP_FORM_RNS_I8;
    c.ksplit = 1;
    if (c.form == MODP_FORM_RNS_I8) {
        // 256x256 tiles while the grid (tiles x moduli) still holds two
        // workgroups per CU
        const int r = rns_planes(g.mp.p, g.k < RNS_KCHUNK ? g.k : RNS_KCHUNK);
        c.tile_m = c.tile_n = tiles_of(g, 256, 256) * r >= 2 * ctx->num_cus ? 256 : 128;
        return c;
    }
    c.tile_m = c.tile_n = 64;
    const int64_t t128 = tiles_of(g, 128, 128);
    if (c.form == MODP_FORM_PLAIN_F64) {
        // 128x128 tiles measured best at n = 8192; a grid of at most one
        // workgroup per CU is cut into concurrent K slices, up to about four
        // workgroups per CU, each at least 256 deep (1024^2: 0.238 ms unsplit,
        // 0.142 / 0.100 / 0.106 ms with 2 / 4 / 8 slices of 64x64 tiles)
        if (t128 >= 2 * ctx->num_cus) c.tile_m = c.tile_n = 128;
        const int64_t t = tiles_of(g, c.tile_m, c.tile_n);
        if (t <= ctx->num_cus && g.k >= 1024) {
            int64_t S = 4 * ctx->num_cus / (t > 0 ? t : 1);
            if (S > 8) S = 8;
            while (S > 1 && g.k / S < 256) --S;
            c.ksplit = (int)S;
        }
        return c;
    }
    // digit form.  One and two digits take 128x128 tiles once there are about
    // three for every four CUs (two digits: 2048^3 52.7 us against 64 with 64x64,
    // 2501 x 1203 x 1777 44.0 against 47.4, but 1024^3, 64 tiles, 26 against
    // 18.9) and K is deep enough for the core to outweigh the epilogue, of which
    // 64x64 keeps four workgroups on a CU (4000 x 4000 x 128, two digits: 34.2
    // us against 41.3 with 128x128); three and four digits gain nothing over 64x64
    // Narrow products would compute padding: up to 64 rows or columns (40,000 x 16
    // x 2000, one digit: 184 us with 128x128, 169 with 64x64), with two digits
    // wherever 128x128 pad a fifth more (192 x 20,000 x 2000 143 and 127, 12,000 x
    // 320 x 700 47 and 40; 420 x 12,000 x 2000, a seventh more, 105 and 103).
    const int L = limb_count(g.mp.p);
    const double pad64 = (double)round_up(g.m, 64) * (double)round_up(g.n, 64);
    const double pad128 = (double)round_up(g.m, 128) * (double)round_up(g.n, 128);
    const bool narrow = std::min(g.m, g.n) <= 64 || (L == 2 && 5 * pad128 >= 6 * pad64);
    if (L <= 2 && g.k > 256 && 4 * t128 >= 3 * ctx->num_cus && !narrow) c.tile_m = c.tile_n = 128;
    // K slices where the tiles leave CUs idle and a slice keeps at least 512 of
    // a long K: the slices' sum costs a launch, about what 1024 of K cost
    // (512 x 512 x 4096, two digits: 45 us unsplit, 24.9 / 26.8 with 4 / 8 slices;
    // 1024^3 18.9 unsplit, 24.6 / 28.0 with 2 / 4)
    const int64_t t = tiles_of(g, c.tile_m, c.tile_n);
    if (g.k >= 2048 && 2 * t <= ctx->num_cus) {
        int64_t S = std::min<int64_t>(ctx->num_cus / (t > 0 ? t : 1), g.k / 512);
        c.ksplit = (int)std::min<int64_t>(S, 8);
    }
    return c;
}

int gemm_run(modp_ctx *ctx, const GemmArgs &g, const GemmConfig &cfg)
{
    if (cfg.form == MODP_FORM_LIMB_I8) return gemm_limb_cfg(ctx, g, cfg);
    if (cfg.form == MODP_FORM_RNS_I8) return gemm_rns_run(ctx, g, cfg.tile_m);
    return gemm_plain_cfg(ctx, g, cfg);
}

int gemm_plain_f64(modp_ctx *ctx, const GemmArgs &g)
{
    return gemm_plain_cfg(ctx, g, gemm_default_config(ctx, g, MODP_FORM_PLAIN_F64));
}

int gemm_small_strided(modp_ctx *ctx, const GemmArgs &g, int64_t count, int64_t sa, int64_t sb, int64_t sc,
                       const GemmSize &last)
{
    return launch_f64_small(ctx, g, f64_reduce_interval(g.mp.p), count, sa, sb, sc, last);
}

int gemm_limb_i8(modp_ctx *ctx, const GemmArgs &g)
{
    return gemm_limb_cfg(ctx, g, gemm_default_config(ctx, g, MODP_FORM_LIMB_I8));
}

int gemm_rns_i8(modp_ctx *ctx, const GemmArgs &g)
{
    return gemm_run(ctx, g, gemm_default_config(ctx, g, MODP_FORM_RNS_I8));
}

// bytes of the digit planes of a product without K slices
static size_t limb_plane_bytes(const GemmArgs &g, const GemmConfig &cfg)
{
    const int L = limb_count(g.mp.p);
    int tm, tn;
    limb_tile(cfg, L, g.m, g.n, g.k, false, &tm, &tn);
    const int64_t kmax = ((int64_t)2147483647 / ((int64_t)L * 16384)) / LBK * LBK;
    const int64_t kc = g.k < kmax ? g.k : kmax;
    const int64_t Kp = round_up(kc > 0 ? kc : 1, LBK);
    return (size_t)L * (size_t)(round_up(g.m, tm) + round_up(g.n, tn)) * (size_t)Kp;
}

// the least that the product needs, in 64 x 64 tiles
size_t gemm_limb_scratch_bytes(const GemmArgs &g)
{
    GemmConfig cfg;
    cfg.tile_m = cfg.tile_n = 64;
    return limb_plane_bytes(g, cfg);
}

int gemm_limb_i8_in(modp_ctx *ctx, const GemmArgs &g, const LimbScratch &ws)
{
    GemmConfig cfg = gemm_default_config(ctx, g, MODP_FORM_LIMB_I8);
    cfg.ksplit = 1;
    // planes rounded up to larger tiles may not fit where those of 64 x 64 do
    if (limb_plane_bytes(g, cfg) > ws.bytes) cfg.tile_m = cfg.tile_n = 64;
    return gemm_limb_cfg(ctx, g, cfg, &ws);
}

namespace {

template <typename T, int V>
int gemv_t(modp_ctx *ctx, int64_t m, int64_t k, const T *A, int64_t lda, const T *x, T *y, const ModP &mp)
{
    const double h = (double)((mp.p + 1) / 2 + 2);
    const double r1 = floor((9007199254740992.0 - (double)mp.p) / (h * h));  // at least 7
    const int cadence = r1 >= 1e6 ? 1000000 / GV_U * GV_U : r1 >= GV_U ? (int)r1 / GV_U * GV_U : 4;
    const int64_t rb = (m + 64 * V - 1) / (64 * V);
    // K slices until the grid holds two workgroups per CU, each wave at least two
    // batches; more than 128 slices cost more to sum than they save (6001 x
    // 7003: 64 us with two to eight workgroups per CU, 300 x 20000 16 us with
    // 64 or 128 slices and 19 with 256, 64 x 70000 26 / 18 / 18 us)
    int64_t S = 2 * (int64_t)ctx->num_cus / rb;
    if (S > k / (4 * 2 * GV_U)) S = k / (4 * 2 * GV_U);
    if (S > 128) S = 128;
    // one slice needs no workspace
    if (S < 1 || (S > 1 && k <= 512 && capturing(ctx))) S = 1;
    const int64_t kslice = round_up(((k > 0 ? k : 1) + S - 1) / S, 4 * GV_U);
    S = k > 0 ? (k + kslice - 1) / kslice : 1;
    // y over x or within A: nothing of y is written before all of both is read
    const bool over = k > 0 && m > 0 && (meet(y, y + m, x, x + k) || meet(y, y + m, A, A + (k - 1) * lda + m));
    // the slices' sum in a launch of its own, which is also the way in a graph:
    // the counts of arrivals would be one more workspace that has to be there
    // when it is captured and to stay
    const bool sum_after = over || (S > 1 && capturing(ctx));
    int32_t *P = nullptr;
    int *arrived = nullptr;
    if (S > 1 || sum_after) {
        int st = MODP_OK;
        P = (int32_t *)ws_get(ctx, WS_SLICES, sizeof(int32_t) * (size_t)S * (size_t)m, &st);
        if (!P) return st;
    }
    if (S > 1 && !sum_after) {
        int st = MODP_OK;
        const size_t had = ctx->ws_size[WS_GEMV];
        arrived = (int *)ws_get(ctx, WS_GEMV, sizeof(int) * (size_t)rb, &st);
        if (!arrived) return st;
        if (ctx->ws_size[WS_GEMV] != had) {
            const int n = (int)(ctx->ws_size[WS_GEMV] / sizeof(int));
            k_zero_ints<<<(n + 255) / 256, 256, 0, ctx->stream>>>(arrived, n);
            HIP_TRY(ctx, hipGetLastError());
        }
    }
    {
        TimedLaunch tl(ctx, "gemv");
        k_gemv<T, V><<<dim3((unsigned)rb, (unsigned)S), 256, 0, ctx->stream>>>(m, k, A, lda, x, y, P, arrived, kslice,
                                                                               cadence, mp);
        HIP_TRY(ctx, hipGetLastError());
    }
    if (!sum_after) return MODP_OK;
    GemmArgs g;
    g.m = m; g.n = 1; g.k = k;
    g.C = y; g.ldc = m; g.kc = sizeof(T) == 8 ? EK_F64 : EK_F32;
    g.epi = EPI_STORE;
    g.mp = mp;
    return launch_slice_sum(ctx, g, EPI_STORE, P, (int)S);
}

}  // namespace

int gemv_run(modp_ctx *ctx, int kind, int64_t m, int64_t k, const void *A, int64_t lda, const void *x, void *y,
             int64_t p)
{
    if (m <= 0) return MODP_OK;
    const ModP mp = make_modp(p);
    if (kind == EK_F64) {
        if (m < 2) return gemv_t<double, 1>(ctx, m, k, (const double *)A, lda, (const double *)x, (double *)y, mp);
        return gemv_t<double, 2>(ctx, m, k, (const double *)A, lda, (const double *)x, (double *)y, mp);
    }
    if (m < 4) return gemv_t<float, 1>(ctx, m, k, (const float *)A, lda, (const float *)x, (float *)y, mp);
    return gemv_t<float, 4>(ctx, m, k, (const float *)A, lda, (const float *)x, (float *)y, mp);
}
