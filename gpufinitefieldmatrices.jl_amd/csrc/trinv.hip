// trinv.hip -- inverses mod p: triangular matrices (64-row diagonal blocks
// inverted in LDS, then the off-diagonal blocks by GEMM, level by level, the
// independent products of a small level in one launch) and square matrices
// through PLUQ, A^{-1} = Q U^{-1} L^{-1} P.
//
// Reference: upper/lower_triangular_inverse_no_copy
// (src/CuModMatrix/triangular/triangular_inverse_no_copy.jl:18-478), whose
// recursion splits at a multiple of its tile width and combines with
// X12 = -X11 T12 X22; and inverse / is_invertible_with_inverse
// (src/CuModMatrix/CuModMatrix.jl:351-502), which multiplies the permuted
// triangular inverses.  Inverses are unique, so the split and the GEMM form
// do not change the result.
#include <algorithm>

#include "common.h"

namespace {

constexpr int TB = 64;  // diagonal block edge

typedef double v4d __attribute__((ext_vector_type(4)));

// x - p rint(x / p): at most p/2 + p 2^-22 in magnitude for |x| < 2^53
__device__ __forceinline__ double near_mod(double x, const ModP &mp) { return fma(-rint(x * mp.pinv), mp.pd, x); }

// c + a b over four k, reduced: |products| < 2^50 up to p = 2^26
__device__ __forceinline__ v4d mfma_mod(double a, double b, v4d c, const ModP &mp)
{
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = near_mod(c[e], mp);
    return c;
}

// Inverse of each TB x TB diagonal block of the triangular int32 matrix T
// (k x k, leading dimension ldt) into the same block of X.  One workgroup
// per block; an upper block is worked on as its transpose.  A zero diagonal
// entry sets *bad.
//
// The 64 columns of the four 16 x 16 diagonal blocks are solved by
// substitution, one lane each (16 steps in registers); 32 and 64 follow from
// X21 = -X22 (T21 X11) in FP64 MFMAs, the accumulators of the first product
// (row 4 e + lane / 16 of column lane % 16) being the operand of the second.
// 24 blocks mod 2^26 - 5: 13 us (a 64-step substitution per column, a
// full reduction per product: 260).
template <bool UPPER>
__global__ __launch_bounds__(256) void k_trinv_diag(const int32_t *__restrict__ T, int64_t ldt,
                                                    int32_t *__restrict__ X, int64_t ldx, int64_t k, ModP mp,
                                                    int *__restrict__ bad)
{
    constexpr int P = TB + 1;
    __shared__ double S[TB][P];   // the lower triangle, balanced; identity past the block
    __shared__ double Xs[TB][P];  // its inverse
    __shared__ double dinv[TB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, cl = lane & 15, g = lane >> 4;
    const int64_t o = (int64_t)blockIdx.x * TB;
    const int nb = (int)(k - o < TB ? k - o : TB);
    int32_t v[TB * TB / 256];
#pragma unroll
    for (int i = 0; i < TB * TB / 256; ++i)
        v[i] = T[o + min(lane, nb - 1) + (o + min(wave + 4 * i, nb - 1)) * ldt];
#pragma unroll
    for (int i = 0; i < TB * TB / 256; ++i) {
        const int r = UPPER ? wave + 4 * i : lane, c = UPPER ? lane : wave + 4 * i;
        const int x = v[i] > mp.half ? v[i] - (int)mp.p32 : v[i];
        S[r][c] = r < nb && c < nb ? (r >= c ? (double)x : 0.0) : (r == c ? 1.0 : 0.0);
        Xs[r][c] = 0.0;
    }
    __syncthreads();
    if (tid < TB) {
        const double d = S[tid][tid];
        const uint32_t di = d != 0.0 ? modinv((uint32_t)(d < 0.0 ? d + mp.pd : d), mp) : 0u;
        dinv[tid] = (double)((int)di > mp.half ? (int)di - (int)mp.p32 : (int)di);
        if (!di) *bad = 1;
    }
    __syncthreads();
    if (tid < TB) {
        const int o16 = lane & 48;
        double x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = r == cl ? 1.0 : 0.0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = near_mod(near_mod(x[r], mp) * dinv[o16 + r], mp);
#pragma unroll
            for (int q = r + 1; q < 16; ++q) {
                x[q] = fma(-S[o16 + q][o16 + r], x[r], x[q]);
                if ((r & 3) == 3) x[q] = near_mod(x[q], mp);  // four products below 2^50
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) Xs[o16 + r][o16 + cl] = x[r];
    }
    __syncthreads();
    if (wave < 2) {
        // 16 -> 32: rows 32 wave + 16 .., columns 32 wave ..
        const int c0 = 32 * wave, r0 = c0 + 16;
        v4d t = {0.0, 0.0, 0.0, 0.0}, x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int e = 0; e < 4; ++e) t = mfma_mod(S[r0 + cl][c0 + 4 * e + g], Xs[c0 + 4 * e + g][c0 + cl], t, mp);
#pragma unroll
        for (int e = 0; e < 4; ++e) x = mfma_mod(Xs[r0 + cl][r0 + 4 * e + g], t[e], x, mp);
#pragma unroll
        for (int e = 0; e < 4; ++e) Xs[r0 + 4 * e + g][c0 + cl] = -x[e];
    }
    __syncthreads();
    if (wave < 2) {
        // 32 -> 64: rows 32 .., columns 16 wave ..
        v4d t[2], x[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            t[a] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 8; ++q)
                t[a] = mfma_mod(S[32 + 16 * a + cl][4 * q + g], Xs[4 * q + g][16 * wave + cl], t[a], mp);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            x[a] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 8; ++q)
                x[a] = mfma_mod(Xs[32 + 16 * a + cl][32 + 4 * q + g], t[q >> 2][q & 3], x[a], mp);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) Xs[32 + 16 * a + 4 * e + g][16 * wave + cl] = -x[a][e];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TB * TB / 256; ++i) {
        const int j = wave + 4 * i;
        const double x = UPPER ? Xs[j][lane] : Xs[lane][j];
        if (lane < nb && j < nb) X[o + lane + (o + j) * ldx] = (int32_t)(x < 0.0 ? x + mp.pd : x);
    }
}

int64_t rup64(int64_t x) { return (x + 63) / 64 * 64; }

GemmArgs i32_gemm(int64_t m, int64_t n, int64_t k, const int32_t *A, int64_t lda, const int32_t *B, int64_t ldb,
                  int32_t *C, int64_t ldc, int epi, const ModP &mp)
{
    GemmArgs g;
    g.m = m; g.n = n; g.k = k;
    g.A = A; g.lda = lda; g.ka = EK_I32;
    g.B = B; g.ldb = ldb; g.kb = EK_I32;
    g.C = C; g.ldc = ldc; g.kc = EK_I32;
    g.epi = epi;
    g.mp = mp;
    return g;
}

// Off-diagonal blocks of X = T^{-1}, bottom-up by levels, after the diagonal
// blocks are in place and X is zero elsewhere.  At level b the blocks
// [lo, lo + 2b) (lo a multiple of 2b) are completed from their halves:
// upper X12 = -X11 (T12 X22), lower X21 = -X22 (T21 X11), with X11 and X22
// finished at the level below.  The pairs of one level are independent and
// lie at a constant stride: while they are small (b < 512) each of the level's
// two products is one launch over all pairs, the last of which may be cut
// off; larger levels take the automatic form pair by pair.  1500 rows: 88
// launches on side streams were 0.3 ms of an inverse.
int trinv_levels(modp_ctx *ctx, bool upper, const int32_t *T, int64_t ldt, int32_t *X, int64_t ldx, int32_t *tmp,
                 int64_t k, const ModP &mp)
{
    for (int64_t h = TB; h < k; h *= 2) {
        const int64_t count = (k - h + 2 * h - 1) / (2 * h);  // pairs with a second half
        const int64_t rl = std::min(h, k - (2 * (count - 1) * h) - h);  // rows of the last second half
        const bool small = h < 512;
        for (int64_t i = 0; i < (small ? 1 : count); ++i) {
            const int64_t lo = 2 * h * i, n = small ? count : 1, r = small || i + 1 < count ? h : rl;
            const int32_t *T11 = T + lo + lo * ldt;
            int32_t *X11 = X + lo + lo * ldx, *X22 = X11 + h + h * ldx;
            const int64_t st = 2 * h * (1 + ldt), sx = 2 * h * (1 + ldx);  // from pair to pair
            GemmArgs g1, g2;
            GemmSize l1, l2;  // of the last pair
            if (upper) {
                // tmp (h x r) = T12 X22; X12 = 0 - X11 tmp
                g1 = i32_gemm(h, r, r, T11 + h * ldt, ldt, X22, ldx, tmp, h, EPI_STORE, mp);
                g2 = i32_gemm(h, r, h, X11, ldx, tmp, h, X11 + h * ldx, ldx, EPI_SUB, mp);
                l1 = GemmSize{h, rl, rl};
                l2 = GemmSize{h, rl, h};
            } else {
                // tmp (r x h) = T21 X11; X21 = 0 - X22 tmp
                const int64_t ldm = small ? h : r;
                g1 = i32_gemm(r, h, h, T11 + h, ldt, X11, ldx, tmp, ldm, EPI_STORE, mp);
                g2 = i32_gemm(r, h, r, X22, ldx, tmp, ldm, X11 + h, ldx, EPI_SUB, mp);
                l1 = GemmSize{rl, h, h};
                l2 = GemmSize{rl, h, rl};
            }
            if (small) {
                // each pair has its own h x h slice of the temporary
                MODP_TRY(gemm_small_strided(ctx, g1, n, st, sx, h * h, l1));
                MODP_TRY(gemm_small_strided(ctx, g2, n, sx, h * h, sx, l2));
            } else {
                for (const GemmArgs *g : {&g1, &g2})
                    MODP_TRY(gemm_run(ctx, *g, gemm_default_config(ctx, *g, MODP_FORM_AUTO)));
            }
        }
    }
    return MODP_OK;
}

int zero2d(modp_ctx *ctx, void *X, int64_t ldx, size_t es, int64_t rows, int64_t cols)
{
    if (rows <= 0 || cols <= 0) return MODP_OK;
    return hip_check(ctx, hipMemset2DAsync(X, (size_t)ldx * es, 0, (size_t)rows * es, (size_t)cols, ctx->stream),
                     "hipMemset2DAsync");
}

size_t elem_size(int kind) { return kind == EK_F64 ? 8 : 4; }

}  // namespace

// X (k x k int32 in a workspace of k columns of ldx) = inverse of the triangular k x k
// int32 matrix T; entries of T outside the triangle are ignored.  unit: the diagonal
// is known to be ones, so nothing has to be read back (rref of 5 x 7 123 -> 105 us).
int trinv_i32(modp_ctx *ctx, bool upper, const int32_t *T, int64_t ldt, int32_t *X, int64_t ldx, int64_t k,
              const ModP &mp, bool unit)
{
    int st = MODP_OK;
    int *bad = (int *)ws_get(ctx, WS_TRI_FLAG, 64, &st);
    if (!bad) return st;
    // a level's products: h x r at most k^2 / 4, or slices of h^2 for h <= 256
    int32_t *tmp = (int32_t *)ws_get(ctx, WS_TRI_TMP, sizeof(int32_t) * ((size_t)((k + 1) / 2 + TB) * (size_t)(k + TB) + 65536),
                                     &st);
    if (!tmp) return st;
    HIP_TRY(ctx, hipMemsetAsync(X, 0, sizeof(int32_t) * (size_t)ldx * (size_t)k, ctx->stream));
    if (!unit) HIP_TRY(ctx, hipMemsetAsync(bad, 0, sizeof(int), ctx->stream));
    const unsigned nbk = (unsigned)((k + TB - 1) / TB);
    if (upper) k_trinv_diag<true><<<nbk, 256, 0, ctx->stream>>>(T, ldt, X, ldx, k, mp, bad);
    else k_trinv_diag<false><<<nbk, 256, 0, ctx->stream>>>(T, ldt, X, ldx, k, mp, bad);
    HIP_TRY(ctx, hipGetLastError());
    if (unit) return trinv_levels(ctx, upper, T, ldt, X, ldx, tmp, k, mp);
    int hbad = 0;
    HIP_TRY(ctx, hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (hbad)
        return set_error(ctx, MODP_ERR_NOT_INVERTIBLE, "triangular matrix has a zero (or non-invertible) diagonal entry modulo %lld",
                         (long long)mp.p);
    return trinv_levels(ctx, upper, T, ldt, X, ldx, tmp, k, mp);
}

int tri_inverse(modp_ctx *ctx, int kind, int upper, int64_t m, int64_t n, const void *A, int64_t lda, void *Ainv,
                int64_t ldai, int64_t p)
{
    if (!upper && m > n)
        return set_error(ctx, MODP_ERR_DIM, "(Right) pseudoinverse not defined for tall lower triangular matrices");
    const int64_t k = m < n ? m : n;
    // Ainv is n x m: the leading k x k block holds the inverse, zeros elsewhere
    MODP_TRY(zero2d(ctx, Ainv, ldai, elem_size(kind), n, m));
    if (k == 0) return MODP_OK;
    const ModP mp = make_modp(p);
    const int64_t ld = rup64(k);
    int st = MODP_OK;
    int32_t *T = (int32_t *)ws_get(ctx, WS_TRI_T, sizeof(int32_t) * (size_t)ld * (size_t)k, &st);
    if (!T) return st;
    int32_t *X = (int32_t *)ws_get(ctx, WS_TRI_X, sizeof(int32_t) * (size_t)ld * (size_t)k, &st);
    if (!X) return st;
    MODP_TRY(util_convert(ctx, kind, k, k, A, lda, EK_I32, T, ld, mp));
    MODP_TRY(trinv_i32(ctx, upper != 0, T, ld, X, ld, k, mp));
    return util_convert(ctx, EK_I32, k, k, X, ld, kind, Ainv, ldai, mp);
}

int mat_inverse(modp_ctx *ctx, int form, int kind, int64_t n, const void *A, int64_t lda, void *Ainv, int64_t ldai,
                int64_t p, int *invertible)
{
    *invertible = 0;
    if (n == 0) {
        *invertible = 1;
        return MODP_OK;
    }
    int taken = 0;
    MODP_TRY(elim_inverse(ctx, form, kind, n, A, lda, Ainv, ldai, p, invertible, &taken));
    if (taken) return MODP_OK;
    const ModP mp = make_modp(p);
    const int64_t ld = rup64(n);
    const size_t es = elem_size(kind);
    int st = MODP_OK;
    void *U = ws_get(ctx, WS_INV_U, es * (size_t)ld * (size_t)n, &st);
    if (!U) return st;
    void *L = ws_get(ctx, WS_INV_L, es * (size_t)ld * (size_t)n, &st);
    if (!L) return st;
    // (the elimination writes all n rows and columns of both)
    ElimResult r;
    MODP_TRY(elim_run(ctx, ELIM_PLUQ, form, kind, n, n, A, lda, U, ld, L, ld, p, r));
    if (r.rank < n) return MODP_OK;
    *invertible = 1;
    // U^{-1} and L^{-1} as int32, in the triangular workspaces' places
    int32_t *T = (int32_t *)ws_get(ctx, WS_TRI_T, sizeof(int32_t) * (size_t)ld * (size_t)n, &st);
    if (!T) return st;
    int32_t *Xu = (int32_t *)ws_get(ctx, WS_TRI_X, sizeof(int32_t) * (size_t)ld * (size_t)n, &st);
    if (!Xu) return st;
    int32_t *Xl = (int32_t *)ws_get(ctx, WS_TRI_X2, sizeof(int32_t) * (size_t)ld * (size_t)n, &st);
    if (!Xl) return st;
    MODP_TRY(util_convert(ctx, kind, n, n, U, ld, EK_I32, T, ld, mp));
    MODP_TRY(trinv_i32(ctx, true, T, ld, Xu, ld, n, mp, true));
    MODP_TRY(util_convert(ctx, kind, n, n, L, ld, EK_I32, T, ld, mp));
    MODP_TRY(trinv_i32(ctx, false, T, ld, Xl, ld, n, mp));
    // A^{-1} = Q U^{-1} L^{-1} P: apply_row_inv_perm!(col stack, U^{-1}) and
    // apply_col_inv_perm!(row stack, L^{-1}), then the product
    MODP_TRY(util_perm(ctx, EK_I32, 1, n, n, Xu, ld, r.col_swaps.data(), (int64_t)r.col_swaps.size() / 2, 1));
    MODP_TRY(util_perm(ctx, EK_I32, 0, n, n, Xl, ld, r.row_swaps.data(), (int64_t)r.row_swaps.size() / 2, 1));
    GemmArgs g;
    g.m = n; g.n = n; g.k = n;
    g.A = Xu; g.lda = ld; g.ka = EK_I32;
    g.B = Xl; g.ldb = ld; g.kb = EK_I32;
    g.C = Ainv; g.ldc = ldai; g.kc = kind;
    g.epi = EPI_STORE;
    g.mp = mp;
    GemmConfig cfg = gemm_default_config(ctx, g, form == MODP_FORM_AUTO ? MODP_FORM_AUTO : form);
    return gemm_run(ctx, g, cfg);
}
