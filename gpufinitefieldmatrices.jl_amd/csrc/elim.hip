// elim.hip -- blocked right-looking mod-p elimination on gfx950.
//
// One driver serves pluq (column pivoting of zero columns), lu (PLE: zero
// columns skipped) and rref (PLE followed by blocked back-elimination).  The
// matrix is copied into an int32 working array W (column-major) that keeps L
// and U in place: the pivot of pivot number k sits at row k, column pivcol[k]
// (== k for pluq), the multipliers below it are L's column k, and the
// normalised pivot row is U's row k.
//
// Structure per outer block of NBO columns (reference: the unblocked loop of
// src/CuModMatrix/rref_lu_pluq/pluq_kernels.jl:90-142, one pivot per host
// iteration with a host round-trip each; here one launch factors a whole
// panel):
//   for each inner panel of w <= 32 columns:
//     k_panel    (elim_panel.h) the panel in registers, one row per lane; per
//                column: wave64 argmax by DPP with lowest-row tie-break,
//                across waves through LDS or one XCD's L2, the pivot's
//                inverse, and the rank-1 update of the remaining panel
//                columns; rows move only at the end, by a row map, and
//                the old values of the moved rows in the block's other
//                columns are staged.  Above what an XCD holds at once
//                (16,384 rows) k_panel_g does the same with the panel left in
//                W (any row count).
//     k_update   the block's other columns: the row map, and right of the
//                panel the rows of U (a product with the inverse triangle
//                that the panel leaves) and the rank-w update of every row
//                below the pivots.
//   after the outer block: k_block_finish applies the block's row moves and
//   the solve with the block's L11 to the far columns, then one GEMM with
//   K = NBO (limb or plain form) updates the far trailing block.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "elim_panel.h"

namespace {

constexpr int NBO = 128;  // outer block width (K of the trailing GEMM)

// Panel factorisation for any number of rows (the register panel holds at
// most 16,384 and its keys 2^15 positions): the same outputs as k_panel from
// one 1024-thread workgroup that keeps the panel in W.  Thread t owns local rows t + 1024 q and is the only thread that reads
// or writes them during the column steps; a row's current position (the
// reference's swap of positions pc and Ip) is kept in gpos[row], the row at
// each position in grow[pos].  Per column: the owners scan their eligible
// rows (position >= pc) with 64-bit keys (residue, then lowest position),
// the wave winners publish their rows and inverses in LDS, and after one
// barrier every thread knows the pivot; thread 0 swaps the positions, the
// lanes below w normalise the pivot row, and after a second barrier the
// owners apply the rank-1 update to their rows (residues reduced every
// time).  At the end the moved rows (at most 2 w) go through LDS to their
// positions, the pivot rows with their 1 and normalised U row.
constexpr int GPT = 1024, GNBW = 16;
template <int NBW>
__global__ __launch_bounds__(GPT) void k_panel_g(int32_t *__restrict__ W, int64_t ldw, int m, int kr0_in, int c0,
                                                 int w, ModP mp, int ple, int32_t *__restrict__ ipiv,
                                                 int32_t *__restrict__ pivval, int32_t *__restrict__ pivinv,
                                                 int32_t *__restrict__ pivcol, int32_t *__restrict__ map_dst,
                                                 int32_t *__restrict__ map_src, PanelCtl *__restrict__ ctl,
                                                 int *__restrict__ abort, int KC, int FAR, int32_t *__restrict__ stage,
                                                 int *__restrict__ cursor, int32_t *__restrict__ gpos,
                                                 int32_t *__restrict__ grow, PanelSolve *__restrict__ solve, int strict,
                                                 int *__restrict__ told)
{
    constexpr int NW = GPT / 64;
    if (abort && *abort) {
        if (threadIdx.x == 0) {
            ctl->npiv = 0;
            ctl->status = 4;
            ctl->ncols = 0;
            ctl->nmap = 0;
            ctl->kr0 = kr0_in;
        }
        return;
    }
    const int kr0 = cursor ? *cursor : kr0_in;
    __shared__ uint64_t s_key[NW];
    __shared__ int s_row[NW];
    __shared__ uint32_t s_cinv[NW];
    __shared__ uint32_t s_crow[NW][NBW];
    __shared__ uint32_t s_U[NBW][NBW];
    __shared__ int s_ip[NBW], s_pv[NBW], s_pi[NBW], s_pcol[NBW];
    __shared__ int s_msrc[2 * NBW], s_mdst[2 * NBW];
    __shared__ uint32_t s_mv[2 * NBW][NBW], s_T[NBW][NBW];
    __shared__ int s_cnt, s_num[PNW];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rows = m - kr0;
    int32_t *P = W + kr0 + (int64_t)c0 * ldw;  // local row i, panel column j: P[i + j ldw]
    for (int i = tid; i < rows; i += GPT) {
        gpos[i] = i;
        grow[i] = i;
    }
    if (tid == 0) s_cnt = 0;
    __syncthreads();

    int pc = 0, status = 0, consumed = w;
    bool active = true;
    for (int jc = 0; jc < NBW; ++jc) {
        const bool run = active && jc < w && pc < rows;
        if (active && jc < w && pc >= rows) {
            status = 2;
            consumed = jc;
            active = false;
        }
        uint64_t mine = 0;
        int mrow = -1;
        if (run) {
            for (int i = tid; i < rows; i += GPT) {
                const int ps = gpos[i];
                if (ps < pc) continue;
                const uint32_t v = (uint32_t)P[i + (int64_t)jc * ldw];
                const uint64_t k = ((uint64_t)v << 32) | (uint32_t)(0x7fffffff - ps);
                if (v != 0 && k > mine) {
                    mine = k;
                    mrow = i;
                }
            }
        }
        const uint64_t wbest = wave_max(mine);
        if (mine != 0 && mine == wbest) {
            // keys are unique: one lane per wave publishes its row
            const uint32_t V = (uint32_t)(mine >> 32);
            s_key[wave] = mine;
            s_row[wave] = mrow;
            s_cinv[wave] = modinv_fast(V, mp);
            for (int j = jc + 1; j < NBW; ++j) s_crow[wave][j] = j < w ? (uint32_t)P[mrow + (int64_t)j * ldw] : 0u;
        }
        if (lane == 0 && wbest == 0) s_key[wave] = 0;
        __syncthreads();
        uint64_t best = s_key[0];
        int bw = 0;
        for (int x = 1; x < NW; ++x) {
            const uint64_t k = s_key[x];
            if (k > best) {
                best = k;
                bw = x;
            }
        }
        const uint32_t V = (uint32_t)(best >> 32);
        const int Ip = 0x7fffffff - (int)(uint32_t)best;
        const uint32_t inv = V != 0 ? s_cinv[bw] : 0u;
        const int wrow = V != 0 ? s_row[bw] : -1;
        const bool piv = run && V != 0 && inv != 0;
        if (run && V == 0) {
            if (!ple) {
                status = 1;
                consumed = jc;
                active = false;
            }
        }
        if (run && V != 0 && inv == 0) {
            status = 3;
            consumed = jc;
            active = false;
        }
        if (piv) {
            if (tid == 0) {
                // the winner moves to position pc, the row at pc to Ip
                const int rpc = grow[pc];
                gpos[wrow] = pc;
                gpos[rpc] = Ip;
                grow[Ip] = rpc;
                grow[pc] = wrow;
                s_ip[pc] = Ip;
                s_pv[pc] = (int)V;
                s_pi[pc] = (int)inv;
                s_pcol[pc] = jc;
            }
            if (tid > jc && tid < NBW) s_U[pc][tid] = tid < w ? mulmod(s_crow[bw][tid], inv, mp) : 0u;
        }
        __syncthreads();
        if (piv) {
            const int pn = pc + 1;
            for (int i = tid; i < rows; i += GPT) {
                if (gpos[i] < pn) continue;
                const uint32_t l = (uint32_t)P[i + (int64_t)jc * ldw];
                if (l == 0) continue;
                for (int j = jc + 1; j < w; ++j) {
                    int32_t *x = P + i + (int64_t)j * ldw;
                    *x = (int32_t)submod((uint32_t)*x, mulmod(l, s_U[pc][j], mp), mp);
                }
            }
            pc = pn;
        }
        // the next step's LDS writes come after every read of this one
        __syncthreads();
    }

    // Row gather map: positions 0..pc-1 first, in order, then every other
    // row that moved.
    for (int i = tid; i < rows; i += GPT) {
        const int ps = gpos[i];
        if (ps < pc) {
            map_dst[ps] = kr0 + ps;
            map_src[ps] = kr0 + i;
            s_msrc[ps] = i;
            s_mdst[ps] = ps;
        } else if (ps != i) {
            const int e = pc + atomicAdd(&s_cnt, 1);
            map_dst[e] = kr0 + ps;
            map_src[e] = kr0 + i;
            s_msrc[e] = i;
            s_mdst[e] = ps;
        }
    }
    __syncthreads();
    const int nmap_all = pc + s_cnt;
    // old values of the moved rows in the block's other columns
    const int ncol_other = (FAR - KC) - w, nstage = nmap_all * ncol_other;
    for (int idx = tid; idx < nstage; idx += GPT) {
        const int e = idx % nmap_all, ci = idx / nmap_all;
        const int c = ci < c0 - KC ? KC + ci : KC + ci + w;
        stage[e + 64 * ci] = W[(int64_t)kr0 + s_msrc[e] + (int64_t)c * ldw];
    }
    // the moved rows' final panel values, then their stores
    for (int idx = tid; idx < nmap_all * NBW; idx += GPT) {
        const int e = idx % nmap_all, j = idx / nmap_all;
        if (j < w) {
            const int k = s_mdst[e];
            const int jk = k < pc ? s_pcol[k] : NBW;
            s_mv[e][j] = j < jk ? (uint32_t)P[s_msrc[e] + (int64_t)j * ldw] : (j == jk ? 1u : s_U[k][j]);
        }
    }
    __syncthreads();
    for (int idx = tid; idx < nmap_all * NBW; idx += GPT) {
        const int e = idx % nmap_all, j = idx / nmap_all;
        if (j < w) P[s_mdst[e] + (int64_t)j * ldw] = (int32_t)s_mv[e][j];
    }
    if (tid < pc) {
        ipiv[kr0 + tid] = kr0 + s_ip[tid];
        pivval[kr0 + tid] = s_pv[tid];
        pivinv[kr0 + tid] = s_pi[tid];
        pivcol[kr0 + tid] = c0 + s_pcol[tid];
        // column tid of T by substitution, the multipliers from the pivot rows
        for (int t = 0; t < pc; ++t) {
            uint32_t x = t == tid ? 1u : 0u;
            for (int k = tid; k < t; ++k) x = submod(x, mulmod(s_mv[t][s_pcol[k]], s_T[k][tid], mp), mp);
            s_T[t][tid] = t < tid ? 0u : mulmod(x, (uint32_t)s_pi[t], mp);
        }
    }
    if (tid < PNW) s_num[tid] = -1;
    __syncthreads();
    if (tid < pc) s_num[s_pcol[tid]] = tid;
    __syncthreads();
    if (tid < PNW) solve->num[tid] = s_num[tid];
    for (int idx = tid; idx < PNW * PNW; idx += GPT) {
        const int j = idx / PNW, q = idx % PNW, t = s_num[j];
        const uint32_t x = t >= 0 && q < pc ? s_T[t][q] : 0u;
        solve->t[j][q] = x > mp.half ? (int32_t)x - (int32_t)mp.p : (int32_t)x;
    }
    if (tid == 0) {
        ctl->npiv = pc;
        ctl->status = status;
        ctl->ncols = consumed;
        ctl->nmap = nmap_all;
        ctl->kr0 = kr0;
        if (cursor) *cursor = kr0 + pc;
        if (abort && (status != 0 || (strict && pc < w))) {
            *abort = 1;
            tell(told);
        }
    }
}

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d mfma_f64(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// a residue in [0,p) as its balanced representative
__device__ __forceinline__ double balanced(int32_t x, const ModP &mp)
{
    return (double)(x > mp.half ? x - (int32_t)mp.p : x);
}
// EVERY (p > 2^24): four products below 2^50 and a reduced sum stay below
// 2^53, so the sum is reduced after every step; below, up to 128 products
// below 2^46 are summed exactly and reduced once.
template <bool EVERY> __device__ __forceinline__ v4d after_step(v4d c, const ModP &mp)
{
    if (EVERY)
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = near_mod(c[e], mp);
    return c;
}

// The composed row moves of an outer block's panels so far, kept by the updates
// for k_block_finish: the row that is now at position KR + k comes from top[k],
// the one at any other moved position dst[i] from src[i].
struct BlockMoves {
    int32_t n, pad[3];
    int32_t top[NBO], dst[NBO], src[NBO];
};

// After panel t at (kr0, c0, w) of the outer block [KC, FAR), in one launch:
// the panel's row moves for every other column of the block, and for the
// columns right of the panel the rows of U and the rank-npiv update of every
// row below the pivots.  The old values of moved rows come from the stage the
// panel kernel filled before anything moved, so no block reads a row that
// another block writes.
//
// The launch is bound by the latency of its loads, launch and end; the
// arithmetic is two short chains of FP64 MFMAs.  The panel supplies T, the
// inverse of its scaled triangle, so the rows of U are T times the old pivot
// rows instead of a substitution.  A wave takes 32 rows by 16 columns and
// works out its 32 x 16 of U itself: the accumulators of v_mfma_f64_16x16x4
// hold row 4 e + lane / 16 of column lane % 16, which is just the operand of
// the next product's step e, so nothing passes through LDS and no wave waits
// for another; in that product the rows of W run along the lanes (64-byte
// pieces).  Block 0 composes the row moves, the next ones move rows left of
// the panel.  Mean over the panels of a 4096^2 PLUQ mod 65521 8.3 us, of a
// 1500^2 inverse mod 2^26 - 5 7.9 us; with a substitution by one lane per column
// and, above 2^16, a reduction per product 12.7 and 30 us.
constexpr int UT_R = 64, UT_C = 32, UT_L = 8;  // rows, columns of a tile; columns of a block left of the panel
template <bool EVERY>
__global__ __launch_bounds__(256) void k_update(int32_t *__restrict__ W, int64_t ldw, int m, int KR, int KC, int FAR,
                                                int c0, int w, int kr0_in, int first,
                                                const PanelCtl *__restrict__ ctl,
                                                const PanelSolve *__restrict__ solve,
                                                const int32_t *__restrict__ map_dst,
                                                const int32_t *__restrict__ map_src,
                                                const int32_t *__restrict__ stage, BlockMoves *__restrict__ moves,
                                                ModP mp, const int *__restrict__ skip)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nl = c0 - KC, nr = FAR - (c0 + w), gl = (nl + UT_L - 1) / UT_L;
    if (blockIdx.x == 0) {
        // new moves after the old ones: a thread holds the position KR + tid, or
        // one of the others
        __shared__ int s_dst[64], s_src[64], s_from[64];
        __shared__ int s_n;
        const int skipped = skip ? *skip : 0, nmap = ctl->nmap;
        const bool top = tid < NBO;
        const int i = top ? tid : tid - NBO, nold = first ? 0 : moves->n;
        bool keep = top || i < nold;
        const int dst = top ? KR + i : keep ? moves->dst[i] : -1;
        int src = top ? (first ? dst : moves->top[i]) : keep ? moves->src[i] : -1;
        if (tid < 64) {
            s_dst[tid] = map_dst[tid];
            s_src[tid] = s_from[tid] = map_src[tid];
        }
        if (tid == 0) s_n = 0;
        __syncthreads();
        if (skipped) return;
        int at = -1;
        for (int e = 0; e < nmap; ++e) {
            if (keep && s_src[e] == dst) s_from[e] = src;
            if (keep && s_dst[e] == dst) at = e;
        }
        __syncthreads();
        if (top) {
            moves->top[i] = at >= 0 ? s_from[at] : src;
        } else if (keep && at < 0) {
            const int k = atomicAdd(&s_n, 1);
            moves->dst[k] = dst;
            moves->src[k] = src;
        }
        if (tid < nmap && (s_dst[tid] < KR || s_dst[tid] >= KR + NBO)) {
            const int k = atomicAdd(&s_n, 1);
            moves->dst[k] = s_dst[tid];
            moves->src[k] = s_from[tid];
        }
        __syncthreads();
        if (tid == 0) moves->n = s_n;
        return;
    }
    if ((int)blockIdx.x <= gl) {
        const int skipped = skip ? *skip : 0, nmap = ctl->nmap;
        if (skipped) return;
        const int cb = ((int)blockIdx.x - 1) * UT_L, nc = min(UT_L, nl - cb);
        for (int idx = tid; idx < nmap * nc; idx += 256) {
            const int e = idx % nmap, ci = cb + idx / nmap;
            W[(int64_t)map_dst[e] + (int64_t)(KC + ci) * ldw] = stage[e + 64 * ci];
        }
        return;
    }
    // Every load that does not depend on another is issued first, at indices
    // clamped into range; values that are not needed meet a zero of T.
    const int tile = (int)blockIdx.x - 1 - gl, ncg = (nr + UT_C - 1) / UT_C;
    const int cl = lane & 15, g = lane >> 4;
    const int cw = (tile % ncg) * UT_C + (wave >> 1) * 16;  // column right of the panel
    if (cw >= nr) return;
    const int skipped = skip ? *skip : 0;
    const int npiv = ctl->npiv, nmap = ctl->nmap;
    const int kr0 = kr0_in >= 0 ? kr0_in : ctl->kr0;
    const int mdst = map_dst[lane];
    int4 t4[2][2], x4[2];
    const int32_t *xs = stage + 64 * (int64_t)(nl + min(cw + cl, nr - 1)) + 8 * g;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) t4[ti][h] = *(const int4 *)&solve->t[16 * ti + cl][8 * g + 4 * h];
        x4[h] = *(const int4 *)(xs + 4 * h);
    }
    const int rel0 = (tile / ncg) * UT_R + (wave & 1) * 32;  // the wave's first row under kr0
    if (skipped || nmap == 0 || kr0 + rel0 >= m) return;
    const int32_t *Lp = W + (int64_t)c0 * ldw;
    int32_t *Cp = W + (int64_t)(c0 + w + cw) * ldw;
    int32_t lv[2][8], cv[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int r = min(kr0 + rel0 + 16 * a + cl, m - 1);
#pragma unroll
        for (int s = 0; s < 8; ++s) lv[a][s] = Lp[r + (int64_t)min(4 * s + g, w - 1) * ldw];
#pragma unroll
        for (int e = 0; e < 4; ++e) cv[a][e] = Cp[r + (int64_t)min(4 * e + g, nr - 1 - cw) * ldw];
    }
    // the rows of the tile that moved here from elsewhere
    __shared__ int s_e[4][32];
    if (lane < 32) s_e[wave][lane] = -1;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int d = mdst - kr0 - rel0;
    if (lane >= npiv && lane < nmap && d >= 0 && d < 32) s_e[wave][d] = lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    int ent[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) ent[a] = s_e[wave][16 * a + cl];
    if (__any(ent[0] >= 0 || ent[1] >= 0)) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ent[a] >= 0) cv[a][e] = stage[ent[a] + 64 * (int64_t)(nl + min(cw + 4 * e + g, nr - 1))];
    }
    // U, rows by panel column
    v4d u[2] = {v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int4 xq = x4[s >> 2];
        const double x = balanced((s & 3) == 0 ? xq.x : (s & 3) == 1 ? xq.y : (s & 3) == 2 ? xq.z : xq.w, mp);
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) {
            const int4 tq = t4[ti][s >> 2];
            const double t = (double)((s & 3) == 0 ? tq.x : (s & 3) == 1 ? tq.y : (s & 3) == 2 ? tq.z : tq.w);
            u[ti] = after_step<EVERY>(mfma_f64(t, x, u[ti]), mp);
        }
    }
    if (!EVERY)
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) u[ti] = after_step<true>(u[ti], mp);
    if (rel0 == 0 && cw + cl < nr) {
        // the pivot rows
        int32_t *dst = Cp + (int64_t)cl * ldw + kr0;
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = solve->num[16 * ti + 4 * e + g];
                if (t >= 0) dst[t] = (int32_t)from_near(u[ti][e], mp);
            }
    }
    if (rel0 + 32 <= npiv) return;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        v4d c = v4d{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 8; ++s) c = after_step<EVERY>(mfma_f64(u[s >> 2][s & 3], balanced(lv[a][s], mp), c), mp);
        const int rel = rel0 + 16 * a + cl;
        if (rel >= npiv && kr0 + rel < m) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (cw + 4 * e + g < nr)
                    Cp[kr0 + rel + (int64_t)(4 * e + g) * ldw] =
                        (int32_t)from_near(near_mod((double)cv[a][e] - c[e], mp), mp);
        }
    }
}

constexpr int MAXPAN = 64;  // inner panels per outer block (NBO / smallest panel width, 2)
constexpr int NBATCH = 8;   // outer blocks enqueued without waiting for the host

// T of the diagonal 32 x 32 triangles of a block's L11 by pivot number, for
// blocks whose panels are not 32 pivots in 32 columns each: one thread a column.
// It replaces the panels' own, and runs only when no update needs them again.
__global__ __launch_bounds__(NBO) void k_block_solve(const int32_t *__restrict__ W, int64_t ldw, int KR, int P,
                                                     const int32_t *__restrict__ pivinv,
                                                     const int32_t *__restrict__ pivcol, ModP mp,
                                                     PanelSolve *__restrict__ solve, const int *__restrict__ skip)
{
    if (skip && *skip) return;
    __shared__ double s_l[NBO][PNW + 1], s_x[NBO][PNW + 1], s_inv[NBO];
    const int tid = threadIdx.x, b0 = tid / PNW * PNW, q = tid % PNW;
    // the rows of the triangles (row b0 + t, pivot q), all loads before the first use
    int32_t l[PNW];
    const int64_t lc = (int64_t)pivcol[KR + min(b0 + q, P - 1)] * ldw;
#pragma unroll
    for (int t = 0; t < PNW; ++t) l[t] = W[KR + min(b0 + t, P - 1) + lc];
    s_inv[tid] = balanced(pivinv[KR + min(tid, P - 1)], mp);
#pragma unroll
    for (int t = 0; t < PNW; ++t) s_l[b0 + t][q] = balanced(l[t], mp);
    __syncthreads();
    for (int t = 0; t < PNW; ++t) {
        double x = t == q ? 1.0 : 0.0;
        for (int k = q; k < t; ++k) x = near_mod(fma(-s_l[b0 + t][k], s_x[tid][k], x), mp);
        x = b0 + t < P && t >= q ? near_mod(x * s_inv[b0 + t], mp) : 0.0;
        s_x[tid][t] = x;
        solve[tid / PNW].t[t][q] = (int32_t)x;
    }
}

// End of an outer block with P pivots (rows [KR, KR+P)): the columns outside
// the block [KC, FAR) get its row moves, those right of it also the solve with
// the block's L11, and their U rows go to Ubig (rows 0..consumed-1 by block
// column, zero for block columns without a pivot).
//
// A wave takes 16 columns.  The moved rows are single elements of W far apart
// in a column (up to 2 x 128 lines of 64 bytes a column, read and written),
// which bounds the launch from below; the solve goes 32 pivots at a time, X_i
// = A_i - sum_j<i L_ij U_j and U_i = T_i X_i with T from the panels, in FP64
// MFMAs whose accumulators are the next product's operands as they are.
// DENSE: the pivots are the block's first P columns.  Mean over the blocks of a
// 4096^2 PLUQ mod 65521 21.5 us, of a 1500^2 inverse mod 2^26 - 5 25 us; with the
// panels' moves one after another and a 128-step substitution by lanes 46 and 53.
template <bool EVERY, bool DENSE>
__global__ __launch_bounds__(64) void k_block_finish(int32_t *__restrict__ W, int64_t ldw, int m, int64_t n, int KR,
                                                     int KC, int FAR, int P, int consumed, int gleft,
                                                     const BlockMoves *__restrict__ moves,
                                                     const PanelSolve *__restrict__ solve,
                                                     const int32_t *__restrict__ pivcol,
                                                     int32_t *__restrict__ Ubig, int64_t ldub, ModP mp,
                                                     const int *__restrict__ skip)
{
    if (skip && *skip) return;
    const int lane = threadIdx.x, cl = lane & 15, g = lane >> 4;
    const bool left = (int)blockIdx.x < gleft;
    const int64_t cb = left ? (int64_t)blockIdx.x * 16 : FAR + (int64_t)((int)blockIdx.x - gleft) * 16;
    const int nc = (int)min((int64_t)16, (left ? KC : n) - cb);
    int32_t *const col = W + (cb + min(cl, nc - 1)) * ldw;
    constexpr int NT = NBO / 16;
    // position 16 b + 4 e + g of the block's rows, and the other moved rows
    int32_t x[NT][4], y[2][16];
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = moves->top[16 * b + 4 * e + g];
    const int nrest = moves->n;
    int rs[2], rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        rs[h] = moves->src[lane + 64 * h];
        rd[h] = moves->dst[lane + 64 * h];
    }
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = col[min(x[b][e], m - 1)];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (lane + 64 * h < nrest)
#pragma unroll
            for (int q = 0; q < 16; ++q) y[h][q] = W[rs[h] + (cb + min(q, nc - 1)) * ldw];
    auto store_moved = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (lane + 64 * h < nrest)
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    if (q < nc) W[rd[h] + (cb + q) * ldw] = y[h][q];
        if (cl >= nc) return;
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = 16 * b + 4 * e + g;
                if ((left || k >= P) && KR + k < m) col[KR + k] = x[b][e];
            }
    };
    if (left) {
        store_moved();
        return;
    }
    int64_t lc[NT - 2][4];  // columns of the pivots
#pragma unroll
    for (int b = 0; b < NT - 2; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = min(16 * b + 4 * e + g, P - 1);
            lc[b][e] = (DENSE ? KC + k : pivcol[KR + k]) * ldw;
        }
    v4d u[NT];
#pragma unroll
    for (int i = 0; i < NT / 2; ++i) {
        if (32 * i >= P) {
            u[2 * i] = u[2 * i + 1] = v4d{0, 0, 0, 0};
            continue;
        }
        v4d s[2], r[2] = {v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}};
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            s[a] = v4d{0, 0, 0, 0};
            const int32_t *Lp = W + min(KR + 32 * i + 16 * a + cl, m - 1);
#pragma unroll
            for (int b = 0; b < 2 * i; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s[a] = after_step<EVERY>(mfma_f64(balanced(Lp[lc[b][e]], mp), u[b][e], s[a]), mp);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[a][e] = near_mod(balanced(x[2 * i + a][e], mp) - s[a][e], mp);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    r[a] = after_step<EVERY>(mfma_f64((double)solve[i].t[16 * a + cl][16 * b + 4 * e + g], s[b][e], r[a]), mp);
            u[2 * i + a] = after_step<true>(r[a], mp);
        }
    }
    store_moved();
    if (cl >= nc) return;
    int32_t *ucol = Ubig + (cb + cl - KC) * ldub;
    if (!DENSE) {
        for (int j = g; j < consumed; j += 4) ucol[j] = 0;
        __threadfence_block();
    }
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 16 * b + 4 * e + g;
            if (k < P) {
                const int32_t v = (int32_t)from_near(u[b][e], mp);
                col[KR + k] = v;
                ucol[DENSE ? k : pivcol[KR + k] - KC] = v;
            }
        }
}

// any nonzero in W[r0:m, c0:n] -> *flag = 1
__global__ void k_any_nonzero(const int32_t *__restrict__ W, int64_t ldw, int64_t r0, int64_t m, int64_t c0,
                              int64_t n, int *flag)
{
    const int64_t rows = m - r0, total = rows * (n - c0);
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = r0 + e % rows, j = c0 + e / rows;
        if (W[i + j * ldw] != 0) *flag = 1;
    }
}

template <typename TU>
__global__ void k_extract_u(int64_t m, int64_t n, const int32_t *__restrict__ W, int64_t ldw, int rank,
                            const int32_t *__restrict__ pivcol, TU *__restrict__ U, int64_t ldu)
{
    const int64_t total = m * n;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % m, c = e / m;
        uint32_t v = 0;
        if (r < rank && c >= pivcol[r]) v = (uint32_t)W[r + c * ldw];
        U[r + c * ldu] = from_res<TU>(v);
    }
}

template <typename TL>
__global__ void k_extract_l(int64_t m, const int32_t *__restrict__ W, int64_t ldw, int rank,
                            const int32_t *__restrict__ pivcol, const int32_t *__restrict__ pivval,
                            TL *__restrict__ L, int64_t ldl)
{
    const int64_t total = m * m;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % m, j = e / m;
        uint32_t v = 0;
        if (j < rank) {
            if (r == j) v = (uint32_t)pivval[j];
            else if (r > j) v = (uint32_t)W[r + (int64_t)pivcol[j] * ldw];
        }
        L[r + j * ldl] = from_res<TL>(v);
    }
}

// G[i, j] = W[i, cols[j]] for i < rows, j < nb, zero left of a row's pivot
__global__ void k_gather_cols(const int32_t *__restrict__ W, int64_t ldw, int64_t rows,
                              const int32_t *__restrict__ pivcol, const int32_t *__restrict__ cols, int64_t nb,
                              int32_t *__restrict__ G, int64_t ldg)
{
    const int64_t total = rows * nb;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = e % rows, j = e / rows;
        const int c = cols[j];
        G[i + j * ldg] = c >= pivcol[i] ? W[i + (int64_t)c * ldw] : 0;
    }
}

// the columns that are no pivots' into free_cols, and what each of the n columns
// is: the number of its pivot, or -1 - its place in free_cols
__global__ void k_column_kinds(const int32_t *__restrict__ pivcol, int rank, int n, int32_t *__restrict__ kinds,
                               int32_t *__restrict__ free_cols)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    int lo = 0, hi = rank;  // the first pivot column that is not below c
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (pivcol[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    const bool piv = lo < rank && pivcol[lo] == c;
    kinds[c] = piv ? lo : -1 - (c - lo);
    if (!piv) free_cols[c - lo] = c;
}

// the reduced echelon form: unit vectors in the pivots' columns, Z elsewhere
// (pivots_only: nothing there)
template <typename T>
__global__ void k_write_rref(int64_t m, int64_t n, int rank, const int32_t *__restrict__ kinds, bool pivots_only,
                             const int32_t *__restrict__ Z, int64_t ldz, T *__restrict__ R, int64_t ldr)
{
    const int64_t total = m * n;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % m, c = e / m;
        const int k = kinds[c];
        if (k < 0 && pivots_only) continue;
        const uint32_t v = k >= 0 ? (uint32_t)(r == k) : r < rank ? (uint32_t)Z[r + (int64_t)(-1 - k) * ldz] : 0u;
        R[r + c * ldr] = from_res<T>(v);
    }
}

// nf of the other columns
template <typename T>
__global__ void k_write_free(int64_t m, int64_t nf, int rank, const int32_t *__restrict__ free_cols,
                             const int32_t *__restrict__ Z, int64_t ldz, T *__restrict__ R, int64_t ldr)
{
    const int64_t total = m * nf;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % m, j = e / m;
        R[r + free_cols[j] * ldr] = from_res<T>(r < rank ? (uint32_t)Z[r + j * ldz] : 0u);
    }
}

unsigned grid_for(int64_t total, int64_t cap = 16384)
{
    int64_t b = (total + 255) / 256;
    if (b > cap) b = cap;
    if (b < 1) b = 1;
    return (unsigned)b;
}

int64_t rup(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

// before a batch of blocks: no abort, nothing lost, the first row, nobody arrived
__global__ void k_blocks_begin(int *abort, int *lost, int *cursor, int row, uint32_t *arrive, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        *abort = 0;
        *lost = 0;
        *cursor = row;
    }
    if (i < n) arrive[i] = 0;
}

// the identity, with the rows of padding
__global__ void k_identity(int32_t *__restrict__ W, int64_t ldw, int64_t n)
{
    const int64_t total = ldw * n;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x)
        W[e] = e % ldw == e / ldw;
}

// t[a] = a^{-1} mod p for a < n, 0 where there is none
__global__ void k_inv_table(uint32_t *__restrict__ t, int n, ModP mp)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < n) t[a] = a > 0 && a < mp.p ? modinv_fast((uint32_t)a, mp) : 0u;
}

// Inverses of the residues below PINV (1 MiB at most, 8 us to build), from which
// the panels make every other inverse; built once per modulus and kept in the
// context.
const uint32_t *inverse_table(modp_ctx *ctx, const ModP &mp, int *st)
{
    if (ctx->invtab && ctx->invtab_p == mp.p) return ctx->invtab;
    ctx->invtab_prime = mp.p >= 2;
    for (int64_t q = 2; q * q <= mp.p && ctx->invtab_prime; q += q == 2 ? 1 : 2) ctx->invtab_prime = mp.p % q != 0;
    if (!ctx->invtab) {
        hipError_t e = device_alloc(ctx, (void **)&ctx->invtab, sizeof(uint32_t) * PINV);
        if (e != hipSuccess) { *st = hip_check(ctx, e, "inverse table"); return nullptr; }
    }
    const int n = mp.p < PINV ? (int)mp.p : PINV;
    k_inv_table<<<(n + 255) / 256, 256, 0, ctx->stream>>>(ctx->invtab, n, mp);
    if (hipGetLastError() != hipSuccess) { *st = MODP_ERR_DEVICE; return nullptr; }
    ctx->invtab_p = mp.p;
    return ctx->invtab;
}

}  // namespace

// Rows that the panel on one XCD takes: all of its workgroups (of 256 rows) wait
// for each other, so all have to be on the XCD's CUs at once.  Two fit on a CU
// (75 KB of LDS, at most 231 registers), 64 workgroups or 16,384 rows.
static int64_t panel_rows(modp_ctx *ctx, int arith)
{
    int64_t &rows = ctx->panel_rows[arith];
    if (rows == 0) {
        int n = 0;
        const void *k = arith == 0   ? (const void *)k_panel<true, 0>
                        : arith == 1 ? (const void *)k_panel<true, 1>
                                     : (const void *)k_panel<true, 2>;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, 64 * PWAVES, 0) != hipSuccess) {
            (void)hipGetLastError();
            n = 1;
        }
        const int64_t waves = (int64_t)n * std::min(XCD_CUS, ctx->num_cus) * PWAVES;
        rows = std::max<int64_t>(PSINGLE, 64 * std::min<int64_t>(waves, PXS));
    }
    return rows;
}

// One run from A to the outputs.  meet: panels may go to the workgroups of an
// XCD; *lost: an exchange of theirs did not end, and nothing has been put out.
static int elim_attempt(modp_ctx *ctx, int mode, int form, int kind, int64_t m, int64_t n, const void *A, int64_t lda,
                        void *U, int64_t ldu, void *L, int64_t ldl, int64_t p, ElimResult &res, bool meet, bool *lost)
{
    *lost = false;
    const ModP mp = make_modp(p);
    const bool ple = mode != ELIM_PLUQ;
    const int64_t mn = m < n ? m : n;
    // ELIM_INVERSE: an identity right of the pivot columns
    const int64_t nt = mode == ELIM_INVERSE ? n + m : n;
    res = ElimResult();
    if (m <= 0 || n <= 0) {
        if (mode == ELIM_LU)
            for (int64_t i = 0; i < m; ++i) res.perm.push_back(i + 1);
        if (U && m > 0 && n > 0) return MODP_OK;
        return MODP_OK;
    }
    if (m > (int64_t)1 << 30)
        return set_error(ctx, MODP_ERR_DIM, "elimination supports at most 2^30 rows (got %lld)", (long long)m);

    // Panels of an outer block starting at row KR by the rows left: the register
    // panel of one workgroup (256 rows: one wave per SIMD) or of one XCD, the
    // W-resident panel beyond what an XCD holds (panel_rows).  Mod 65521 a
    // 32-column panel takes 37 us on one workgroup, and on an XCD 45 us up to
    // 4096 rows, 56 at 8192 and 76 at 16,384 (one workgroup with 512 rows, two
    // waves per SIMD: 58 us).  The W-resident panel takes 16,384
    // rows in 0.55 ms for 16 columns.
    // MODP_PANEL_GLOBAL=1 sends every panel to the W-resident kernel (used
    // to compare the two panel kernels at sizes both handle)
    const char *genv = getenv("MODP_PANEL_GLOBAL");
    const bool force_global = genv && atoi(genv) != 0;
    // the cycles that a workgroup of a panel on one XCD waits for the others to
    // start before the panel is left to the W-resident kernel: 2 ms, about what
    // a block takes there (1.6 ms at 4096 rows, 4.4 at 16,384;
    // MODP_PANEL_PATIENCE sets it; below 0 every such panel gives up).  They start together unless other work
    // holds the XCD's CUs, perhaps another context's panel that waits in turn,
    // so after a panel that gave up the W-resident kernel keeps `away` blocks,
    // twice as many each time in a row, and the next try is one block.
    const char *penv = getenv("MODP_PANEL_PATIENCE");
    const long long patience = penv ? atoll(penv) : 5000000LL;
    int away = 0, next_away = 1;
    // MODP_PANEL_SPINS sets how often they look again for a step's words (0: an
    // exchange is lost when one is late, -1: at the first step)
    const char *senv = getenv("MODP_PANEL_SPINS");
    const int spins = senv ? atoi(senv) : EXCHANGE_SPINS;
    const int arith = mp.small ? 0 : mp.p <= ((int64_t)1 << 24) ? 1 : 2;  // of the panels
    auto panel_width = [&](int64_t KR, int away) {
        return force_global || ((away > 0 || !meet) && m - KR > PSINGLE) || m - KR > panel_rows(ctx, arith) ? GNBW : PNW;
    };
    // whether a block's panels met, if it had such panels
    auto met = [&](int64_t KR, int width, bool yes) {
        if (width != PNW || m - KR <= PSINGLE) return;
        away = yes ? 0 : next_away;
        next_away = yes ? 1 : std::min(2 * next_away, 64);
    };

    int st = MODP_OK;
    const int64_t ldw = rup(m, 64);
    int32_t *W = (int32_t *)ws_get(ctx, WS_WORK, sizeof(int32_t) * (size_t)ldw * (size_t)nt, &st);
    if (!W) return st;
    // pivot arrays, per-panel control blocks and row gather maps of one outer block
    const size_t npv = (size_t)mn + 64;
    const size_t piv_bytes = sizeof(int32_t) * (4 * npv + 2 * MAXPAN * 64) + sizeof(PanelCtl) * NBATCH * MAXPAN + 64 +
                             sizeof(uint32_t) * NBATCH * MAXPAN +
                             sizeof(int32_t) * 64 * NBO + sizeof(PanelSolve) * MAXPAN + sizeof(BlockMoves);
    int32_t *piv = (int32_t *)ws_get(ctx, WS_PIV, piv_bytes, &st);
    if (!piv) return st;
    int32_t *ipiv = piv, *pivval = piv + npv, *pivinv = piv + 2 * npv, *pivcol = piv + 3 * npv;
    int32_t *bmap_dst = piv + 4 * npv, *bmap_src = bmap_dst + MAXPAN * 64;
    PanelCtl *bctl = (PanelCtl *)(bmap_src + MAXPAN * 64);  // by block of the batch
    int *flag = (int *)(bctl + NBATCH * MAXPAN);
    int *abort_flag = flag + 1;
    int *lost_flag = flag + 2;
    int *cursor = flag + 3;                         // first row of the next panel (lu, rref)
    uint32_t *arrive = (uint32_t *)(flag + 4);      // one word per panel of the batch
    int32_t *stage = (int32_t *)(arrive + NBATCH * MAXPAN);  // moved rows' old values, 64 x NBO
    PanelSolve *solve = (PanelSolve *)(stage + 64 * NBO);  // one per panel of the block
    BlockMoves *moves = (BlockMoves *)(solve + MAXPAN);
    int32_t *Ubig = (int32_t *)ws_get(ctx, WS_UBUF, sizeof(int32_t) * (size_t)NBO * (size_t)(nt + 1), &st);
    if (!Ubig) return st;
    // row positions of the W-resident panel (position of each row, row at
    // each position)
    int32_t *gpos = nullptr, *grow = nullptr;
    if (force_global || m > PSINGLE) {
        gpos = (int32_t *)ws_get(ctx, WS_GPOS, sizeof(int32_t) * 2 * (size_t)m, &st);
        if (!gpos) return st;
        grow = gpos + m;
    }
    // (what is read back of them, and a word that a panel writes when it stops)
    PanelCtl *hctl = (PanelCtl *)pinned_get(ctx, sizeof(PanelCtl) * NBATCH * MAXPAN + 128, &st);
    if (!hctl) return st;
    int *told = reinterpret_cast<int *>(hctl + NBATCH * MAXPAN) + 16;

    MODP_TRY(util_convert(ctx, kind, m, n, A, lda, EK_I32, W, ldw, mp));
    if (nt > n) {
        k_identity<<<grid_for(ldw * m, 4096), 256, 0, ctx->stream>>>(W + n * ldw, ldw, m);
        HIP_TRY(ctx, hipGetLastError());
    }
    const uint32_t *invs = inverse_table(ctx, mp, &st);
    if (st != MODP_OK) return st;
    // Where the result does not depend on the pivots, the panels may take any
    // (k_panel_any): 15 us a panel at most, against 37 to 53.  Not for a composite
    // modulus, where a pivot without inverse is an error that depends on which
    // one is taken.
    const bool any_pivot = (mode == ELIM_RREF || mode == ELIM_INVERSE) && !force_global && ctx->invtab_prime;
    bool local_moves = true;  // every row moved so far stayed within 64 rows
    // exchange area of the panels on one XCD: its words are recognised by
    // tags that count the context's panels, so old ones are cleared only when
    // the 17 bits of a key's tag (the 31 of a row's) have been through
    PanelExchange *xch = nullptr;
    if (!force_global && m > PSINGLE) {
        const bool fresh = !ctx->ws[WS_PANEL];
        xch = (PanelExchange *)ws_get(ctx, WS_PANEL, sizeof(PanelExchange), &st);
        if (!xch) return st;
        if (fresh) ctx->panel_tag = 0;
    }
    auto next_tag = [&](uint32_t *t) -> int {
        if ((ctx->panel_tag & 0x1ffffu) == 0)
            HIP_TRY(ctx, hipMemsetAsync(xch, 0, (ctx->panel_tag & 0x7fffffffu) == 0 ? sizeof(PanelExchange)
                                                                                     : sizeof(xch->key), ctx->stream));
        *t = ctx->panel_tag;
        ctx->panel_tag += 64;
        return MODP_OK;
    };

    const int64_t pivot_cols = n;
    auto gemm_sub = [&](int64_t r0, int64_t rows, int64_t ca, int64_t cols, int64_t kcol, int64_t K,
                        const int32_t *Ub, const int *skip) -> int {
        if (rows <= 0 || cols <= 0 || K <= 0) return MODP_OK;
        GemmArgs g;
        g.m = rows; g.n = cols; g.k = K;
        g.A = W + r0 + kcol * ldw; g.lda = ldw; g.ka = EK_I32;
        g.B = Ub; g.ldb = NBO; g.kb = EK_I32;
        g.C = W + r0 + ca * ldw; g.ldc = ldw; g.kc = EK_I32;
        g.epi = EPI_SUB;
        g.mp = mp;
        g.skip = skip;
        const int use_form = form != MODP_FORM_AUTO ? form : choose_form(rows, cols, K, p);
        if (use_form == MODP_FORM_LIMB_I8) {
            const int st = gemm_limb_i8(ctx, g);
            if (st != MODP_ERR_OOM || form != MODP_FORM_AUTO) return st;
            ctx->last_error.clear();  // no room for the digit planes
        }
        return gemm_plain_f64(ctx, g);
    };
    auto launch_panel_any = [&](int blk, int t, int64_t KC, int64_t FAR, int64_t rj, int64_t cj, int64_t w) -> int {
        PanelAnyArgs a = {};
        a.W = W; a.ldw = ldw; a.m = (int)m; a.kr0 = (int)rj; a.c0 = (int)cj; a.w = (int)w;
        a.KC = (int)KC; a.FAR = (int)FAR; a.mp = mp; a.invs = invs;
        a.ipiv = ipiv; a.pivcol = pivcol; a.map_dst = bmap_dst + t * 64; a.map_src = bmap_src + t * 64;
        a.stage = stage; a.ctl = bctl + blk * MAXPAN + t; a.solve = solve + t; a.abort = abort_flag; a.told = told;
        TimedLaunch tl(ctx, "elim_panel_any");
        k_panel_any<<<1, 64 * PWAVES, 0, ctx->stream>>>(a);
        return hip_check(ctx, hipGetLastError(), "k_panel_any launch");
    };
    // panel t of block blk of the batch at (rj, cj), width w; it has at most
    // m - rj rows
    auto launch_panel_t = [&](int width, int blk, int t, int64_t KC, int64_t FAR, int64_t rj, int64_t cj, int64_t w,
                              int *abort, int *cursor, bool strict) -> int {
        if (t >= MAXPAN) return set_error(ctx, MODP_ERR_DEVICE, "more than %d panels in an outer block", MAXPAN);
        int32_t *mdst = bmap_dst + t * 64, *msrc = bmap_src + t * 64;
        PanelCtl *pctl = bctl + blk * MAXPAN + t;
        TimedLaunch tl(ctx, width == GNBW ? "elim_panel_global" : m - rj <= PSINGLE ? "elim_panel_one" : "elim_panel_xcd");
        if (width == GNBW) {
            k_panel_g<GNBW><<<1, GPT, 0, ctx->stream>>>(W, ldw, (int)m, (int)rj, (int)cj, (int)w, mp, ple, ipiv,
                                                        pivval, pivinv, pivcol, mdst, msrc, pctl, abort,
                                                        (int)KC, (int)FAR, stage, cursor, gpos, grow, solve + t, strict, told);
            return hip_check(ctx, hipGetLastError(), "k_panel_g launch");
        }
        PanelArgs a = {};
        a.W = W; a.ldw = ldw; a.m = (int)m; a.kr0 = (int)rj; a.c0 = (int)cj; a.w = (int)w; a.ple = ple;
        a.KC = (int)KC; a.FAR = (int)FAR; a.mp = mp; a.invs = invs;
        a.ipiv = ipiv; a.pivval = pivval; a.pivinv = pivinv; a.pivcol = pivcol;
        a.map_dst = mdst; a.map_src = msrc; a.stage = stage; a.ctl = pctl; a.solve = solve + t; a.abort = abort; a.cursor = cursor;
        a.strict = strict;
        a.told = told;
        if (m - rj <= PSINGLE) {
            if (arith == 0) k_panel<false, 0><<<1, PSINGLE, 0, ctx->stream>>>(a);
            else if (arith == 1) k_panel<false, 1><<<1, PSINGLE, 0, ctx->stream>>>(a);
            else k_panel<false, 2><<<1, PSINGLE, 0, ctx->stream>>>(a);
            return hip_check(ctx, hipGetLastError(), "k_panel launch");
        }
        a.x = xch;
        a.arrive = arrive + blk * MAXPAN + t;
        a.G = (int)((m - rj + 255) / 256);
        a.patience = patience;
        a.spins = spins;
        a.lost = lost_flag;
        MODP_TRY(next_tag(&a.tag));
        const unsigned grid = 8 * (a.G - 1) + 1;
        if (arith == 0) k_panel<true, 0><<<grid, 256, 0, ctx->stream>>>(a);
        else if (arith == 1) k_panel<true, 1><<<grid, 256, 0, ctx->stream>>>(a);
        else k_panel<true, 2><<<grid, 256, 0, ctx->stream>>>(a);
        return hip_check(ctx, hipGetLastError(), "k_panel launch");
    };
    auto blocks_begin = [&](int64_t row, int blocks) -> int {
        k_blocks_begin<<<(unsigned)((blocks * MAXPAN + 255) / 256), 256, 0, ctx->stream>>>(
            abort_flag, lost_flag, cursor, (int)row, arrive, blocks * MAXPAN);
        return hip_check(ctx, hipGetLastError(), "k_blocks_begin launch");
    };
    // the control blocks of the batch and the flags after them
    auto read_back = [&]() -> int {
        HIP_TRY(ctx, hipMemcpyAsync(hctl, bctl, sizeof(PanelCtl) * NBATCH * MAXPAN + 3 * sizeof(int),
                                    hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
        *lost = reinterpret_cast<const int *>(hctl + NBATCH * MAXPAN)[2] != 0;
        return MODP_OK;
    };
    // the rest of the outer block [KC, FAR) from row KR after panel t: its row
    // moves, and right of the panel the rows of U and the rank-npiv update below
    // the pivots.  rj is the panel's first row, or (known false) a lower bound with
    // the row on the device
    auto update_t = [&](int blk, int t, bool known, int64_t KR, int64_t KC, int64_t FAR, int64_t rj, int64_t cj, int64_t w,
                        const int *skip) -> int {
        const int64_t nl = cj - KC, nr = FAR - (cj + w);
        if (nl + nr + (nt - (FAR - KC)) == 0) return MODP_OK;
        const int64_t tiles = ((m - rj + UT_R - 1) / UT_R) * ((nr + UT_C - 1) / UT_C);
        const unsigned grid = (unsigned)(1 + (nl + UT_L - 1) / UT_L + tiles);
        const int kr0 = known ? (int)rj : -1;
        TimedLaunch tl(ctx, "elim_update");
        if (mp.p <= ((int64_t)1 << 24))
            k_update<false><<<grid, 256, 0, ctx->stream>>>(W, ldw, (int)m, (int)KR, (int)KC, (int)FAR, (int)cj, (int)w,
                                                           kr0, t == 0, bctl + blk * MAXPAN + t, solve + t, bmap_dst + t * 64,
                                                           bmap_src + t * 64, stage, moves, mp, skip);
        else
            k_update<true><<<grid, 256, 0, ctx->stream>>>(W, ldw, (int)m, (int)KR, (int)KC, (int)FAR, (int)cj, (int)w,
                                                          kr0, t == 0, bctl + blk * MAXPAN + t, solve + t, bmap_dst + t * 64,
                                                          bmap_src + t * 64, stage, moves, mp, skip);
        return hip_check(ctx, hipGetLastError(), "k_update launch");
    };
    // end of an outer block with P pivots over `consumed` columns, found in
    // panels of `width` columns; the multipliers left of it follow the row moves
    // only where somebody reads them (L)
    auto block_end = [&](int64_t KR, int64_t KC, int64_t FAR, int64_t P, int64_t consumed, int width,
                         const int *skip) -> int {
        if (P <= 0) return MODP_OK;
        // columns of the identity that have not met a pivot row yet are left
        // out: while rows move within 64, those from KR + NBO + 64 on
        const int64_t n = mode == ELIM_INVERSE && local_moves ? pivot_cols + std::min(m, KR + NBO + 64) : nt;
        const int64_t gleft = L ? (KC + 15) / 16 : 0, grid = gleft + (n - FAR + 15) / 16;
        if (grid > 0) {
            const bool dense = width == PNW && P == consumed, every = mp.p > ((int64_t)1 << 24);
            if (!dense && n > FAR) {
                k_block_solve<<<1, NBO, 0, ctx->stream>>>(W, ldw, (int)KR, (int)P, pivinv, pivcol, mp, solve, skip);
                HIP_TRY(ctx, hipGetLastError());
            }
            TimedLaunch tl(ctx, "elim_block_finish");
            auto *k = dense ? (every ? k_block_finish<true, true> : k_block_finish<false, true>)
                            : (every ? k_block_finish<true, false> : k_block_finish<false, false>);
            k<<<(unsigned)grid, 64, 0, ctx->stream>>>(W, ldw, (int)m, n, (int)KR, (int)KC, (int)FAR, (int)P,
                                                      (int)consumed, (int)gleft, moves, solve, pivcol, Ubig, NBO, mp,
                                                      skip);
            HIP_TRY(ctx, hipGetLastError());
        }
        const int64_t rbeg = KR + P;
        return gemm_sub(rbeg, m - rbeg, FAR, n - FAR, KC, consumed, Ubig + (FAR - KC) * NBO, skip);
    };

    std::vector<int64_t> col_stack;
    int64_t kr = 0, kc = 0, last = n - 1;
    // careful: block by block, panels that skip zero columns.  A matrix of one block
    // has nothing to enqueue ahead, so LU starts with it
    bool done = false, careful = ple && n <= NBO && !any_pivot;
    // ple: the block met zero columns; if nothing nonzero is left below row
    // kr, no later column has a pivot and the factorisation is complete (rank = kr)
    auto rest_is_zero = [&]() -> int {
        if (kr >= m || kc >= n) return MODP_OK;
        HIP_TRY(ctx, hipMemsetAsync(flag, 0, sizeof(int), ctx->stream));
        k_any_nonzero<<<grid_for((m - kr) * (n - kc), 4096), 256, 0, ctx->stream>>>(W, ldw, kr, m, kc, n, flag);
        HIP_TRY(ctx, hipGetLastError());
        int *hflag = (int *)hctl;
        HIP_TRY(ctx, hipMemcpyAsync(hflag, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
        if (!*hflag) done = true;
        return MODP_OK;
    };
    // an inverse needs a pivot in every column; once one has none the rest is left
    auto singular = [&](int64_t pivots, int64_t columns) { return mode == ELIM_INVERSE && pivots < columns; };
    auto panel_error = [&](const PanelCtl &c) -> int {
        if (c.status == 3)
            return set_error(ctx, MODP_ERR_NOT_INVERTIBLE, "pivot has no inverse modulo %lld (modulus not prime)",
                             (long long)p);
        return MODP_OK;
    };
    // A batch of blocks is enqueued as if every panel of it found a pivot in
    // each of its columns, so that each block's place is known beforehand.  A panel
    // that does not raises the abort flag, which turns the rest of the batch
    // into no-ops, and its block is completed from the host after one
    // synchronization; the host enqueues no further blocks once it sees the word
    // `told` (rref of a 2000^2 matrix of ones 599 -> 349 us, PLUQ 738
    // -> 503).  One a block cost 50 us of an idle GPU each (PLUQ of
    // 4096^2 10.3 ms, in batches of eight 9.8).  After an abort the batches
    // start again from one block, since the next one may be near.
    struct Block {
        int64_t KR, KC, FAR, P;
        int width;
        std::vector<int64_t> rj, cj, w;
    };
    int batch = NBATCH;
    // after a panel that found no pivot among its 64 rows the general panels
    // take `hold` blocks, twice as many each time
    int hold = 0, next_hold = 1;
    while (!done && kr < m && kc < n) {
        std::vector<Block> blocks;
        const bool any = any_pivot && hold == 0;
        {
            int64_t r = kr, c = kc;
            int left = away;
            while ((int)blocks.size() < (hold > 0 ? std::min(hold, batch) : batch) && !careful && r < m) {
                const int64_t colend = ple ? n : last + 1;  // columns usable as pivot columns
                const int64_t nbo = std::min<int64_t>(std::min<int64_t>(colend - c, NBO), any ? m - r : NBO);
                if (nbo <= 0 || (ple && r + nbo > m)) break;
                Block b;
                b.KR = r; b.KC = c; b.FAR = c + nbo; b.P = 0;
                b.width = any ? PNW : panel_width(r, left);
                for (int64_t cj = c; cj < b.FAR && r + b.P < m;) {
                    const int64_t w = std::min(std::min<int64_t>(b.width, b.FAR - cj), m - (r + b.P));
                    b.rj.push_back(r + b.P); b.cj.push_back(cj); b.w.push_back(w);
                    b.P += w;
                    cj += w;
                }
                r += b.P;
                c += b.P;
                blocks.push_back(b);
                if (!any && left-- <= 0 && next_away > 1) break;
            }
        }
        bool stop_zero = false;
        int64_t nbo = 0;
        if (!blocks.empty()) {
            MODP_TRY(blocks_begin(kr, (int)blocks.size()));
            if (!any) {
                local_moves = false;
                hold -= std::min(hold, (int)blocks.size());
                away -= std::min(away, (int)blocks.size());
            }
            __atomic_store_n(told, 0, __ATOMIC_RELAXED);  // (nothing is on its way)
            for (int i = 0; i < (int)blocks.size() && !__atomic_load_n(told, __ATOMIC_RELAXED); ++i) {
                const Block &b = blocks[i];
                for (int t = 0; t < (int)b.w.size(); ++t) {
                    if (any) MODP_TRY(launch_panel_any(i, t, b.KC, b.FAR, b.rj[t], b.cj[t], b.w[t]));
                    else MODP_TRY(launch_panel_t(b.width, i, t, b.KC, b.FAR, b.rj[t], b.cj[t], b.w[t], abort_flag,
                                                 nullptr, true));
                    MODP_TRY(update_t(i, t, true, b.KR, b.KC, b.FAR, b.rj[t], b.cj[t], b.w[t], abort_flag));
                }
                MODP_TRY(block_end(b.KR, b.KC, b.FAR, b.P, b.P, b.width, abort_flag));
            }
            MODP_TRY(read_back());
            if (*lost) return MODP_OK;
            nbo = blocks[0].FAR - blocks[0].KC;
            if (!reinterpret_cast<const int *>(hctl + NBATCH * MAXPAN)[1]) {
                kr = blocks.back().KR + blocks.back().P;
                kc = blocks.back().KC + blocks.back().P;
                batch = std::min(2 * batch, NBATCH);
                if (!any) met(blocks.back().KR, blocks.back().width, true);
            } else {
                int i = 0, t = 0;
                auto full = [&]() {
                    const PanelCtl &c = hctl[i * MAXPAN + t];
                    return c.status == 0 && c.npiv == blocks[i].w[t];
                };
                while (i < (int)blocks.size() && full())
                    if (++t == (int)blocks[i].w.size()) {
                        t = 0;
                        ++i;
                    }
                if (i == (int)blocks.size())
                    return set_error(ctx, MODP_ERR_DEVICE, "elimination pipeline aborted without a stopping panel");
                const Block &b = blocks[i];
                const PanelCtl pc = hctl[i * MAXPAN + t];
                MODP_TRY(panel_error(pc));
                if (pc.status == 5) met(b.KR, b.width, false);
                int64_t P = 0;
                for (int q = 0; q < t; ++q) P += b.w[q];
                const int64_t consumed = P + pc.ncols;
                if (singular(P + pc.npiv, consumed)) break;
                // the update after this panel was skipped by its own flag
                if (pc.npiv > 0) MODP_TRY(update_t(i, t, true, b.KR, b.KC, b.FAR, b.rj[t], b.cj[t], b.w[t], nullptr));
                P += pc.npiv;
                MODP_TRY(block_end(b.KR, b.KC, b.FAR, P, consumed, b.width, nullptr));
                kr = b.KR + P;
                kc = b.KC + consumed;
                nbo = b.FAR - b.KC;
                stop_zero = pc.status == 1;
                batch = 1;
                if (pc.status == 7) {
                    hold = next_hold;
                    next_hold = std::min(2 * next_hold, 64);
                    // the last block is done by panels that skip zero columns at
                    // once: rref of 100^2 with every third column zero 409 -> 376 us
                    careful = mode == ELIM_RREF && b.FAR == n;
                }
                if (P < consumed) {
                    careful = true;
                    MODP_TRY(rest_is_zero());
                }
            }
        } else if (ple) {
            // Panels skip zero columns here, so a panel's first row depends
            // on the pivots found before it.  The panels of the block are
            // enqueued at their fixed columns and each takes its first row
            // from a device cursor that the previous one advanced; the
            // updates read it from the panel's control block.  A panel that
            // runs out of rows (or meets a pivot without inverse) raises the
            // abort flag, which turns the rest of the block into no-ops, and
            // the host reads the outcome once per block.
            const int64_t KR = kr, KC = kc, FAR = KC + std::min<int64_t>(n - KC, NBO);
            const int NBW = panel_width(KR, away);
            away -= std::min(away, 1);
            hold -= std::min(hold, 1);
            local_moves = false;
            nbo = FAR - KC;
            MODP_TRY(blocks_begin(KR, 1));
            std::vector<int64_t> pcj, pw;
            for (int64_t cj = KC; cj < FAR; cj += NBW) {
                pcj.push_back(cj);
                pw.push_back(std::min<int64_t>(NBW, FAR - cj));
            }
            const int np = (int)pcj.size();
            for (int t = 0; t < np; ++t) {
                MODP_TRY(launch_panel_t(NBW, 0, t, KC, FAR, KR, pcj[t], pw[t], abort_flag, cursor, false));
                MODP_TRY(update_t(0, t, false, KR, KC, FAR, KR, pcj[t], pw[t], abort_flag));
            }
            MODP_TRY(read_back());
            if (*lost) return MODP_OK;
            int64_t P = 0, consumed = 0;
            bool gave_up = false;
            for (int t = 0; t < np; ++t) {
                const PanelCtl &pc = hctl[t];
                if (pc.status == 4) break;
                MODP_TRY(panel_error(pc));
                gave_up = pc.status == 5;
                P += pc.npiv;
                consumed += pc.ncols;
                if (pc.status != 0) {
                    // the update after this panel was skipped by its own flag
                    if (pc.npiv > 0) MODP_TRY(update_t(0, t, false, KR, KC, FAR, KR, pcj[t], pw[t], nullptr));
                    break;
                }
            }
            met(KR, NBW, !gave_up);
            if (singular(P, consumed)) break;
            kr += P;
            kc += consumed;
            MODP_TRY(block_end(KR, KC, FAR, P, consumed, NBW, nullptr));
            careful = P < nbo;
            if (P < consumed) MODP_TRY(rest_is_zero());
        }
        if (!ple && kr < m && kc < n && (stop_zero || nbo == 0 || kc > last)) {
            // pluq zero column at kc (rows >= kr zero): whole block zero -> tail,
            // else move it to `last` and retry the same column
            HIP_TRY(ctx, hipMemsetAsync(flag, 0, sizeof(int), ctx->stream));
            k_any_nonzero<<<grid_for((m - kr) * (n - kc), 4096), 256, 0, ctx->stream>>>(W, ldw, kr, m, kc, n, flag);
            HIP_TRY(ctx, hipGetLastError());
            int *hflag = (int *)hctl;
            HIP_TRY(ctx, hipMemcpyAsync(hflag, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
            HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
            if (!*hflag) {
                std::vector<int64_t> tail;
                for (int64_t c = kc; c < n; ++c) {
                    tail.push_back(c + 1);
                    tail.push_back(n);
                    col_stack.push_back(c + 1);
                    col_stack.push_back(n);
                }
                MODP_TRY(util_perm(ctx, EK_I32, 0, m, n, W, ldw, tail.data(), (int64_t)tail.size() / 2, 0));
                done = true;
            } else {
                int64_t sw[2] = {kc + 1, last + 1};
                col_stack.push_back(kc + 1);
                col_stack.push_back(last + 1);
                MODP_TRY(util_perm(ctx, EK_I32, 0, m, n, W, ldw, sw, 1, 0));
                --last;
            }
        }
        if (ple && kr >= m) break;
    }
    const int64_t rank = kr;

    // outputs
    if (U) {
        unsigned g = grid_for(m * n);
        if (kind == EK_F64) k_extract_u<double><<<g, 256, 0, ctx->stream>>>(m, n, W, ldw, (int)rank, pivcol, (double *)U, ldu);
        else k_extract_u<float><<<g, 256, 0, ctx->stream>>>(m, n, W, ldw, (int)rank, pivcol, (float *)U, ldu);
        HIP_TRY(ctx, hipGetLastError());
    }
    if (L && mode != ELIM_RREF) {
        unsigned g = grid_for(m * m);
        if (kind == EK_F64) k_extract_l<double><<<g, 256, 0, ctx->stream>>>(m, W, ldw, (int)rank, pivcol, pivval, (double *)L, ldl);
        else k_extract_l<float><<<g, 256, 0, ctx->stream>>>(m, W, ldw, (int)rank, pivcol, pivval, (float *)L, ldl);
        HIP_TRY(ctx, hipGetLastError());
    }
    std::vector<int32_t> hp((size_t)(2 * (rank > 0 ? rank : 1)));
    if (rank > 0) {
        HIP_TRY(ctx, hipMemcpyAsync(hp.data(), ipiv, sizeof(int32_t) * rank, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(ctx, hipMemcpyAsync(hp.data() + rank, pivcol, sizeof(int32_t) * rank, hipMemcpyDeviceToHost, ctx->stream));
    }
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    res.rank = rank;
    for (int64_t i = 0; i < rank; ++i) {
        if (hp[i] != i) {
            res.row_swaps.push_back(i + 1);
            res.row_swaps.push_back((int64_t)hp[i] + 1);
        }
        res.pivcols.push_back((int64_t)hp[rank + i] + 1);
    }
    res.col_swaps = col_stack;
    if (mode == ELIM_LU) {
        res.perm.resize((size_t)m);
        for (int64_t i = 0; i < m; ++i) res.perm[i] = i + 1;
        for (int64_t i = 0; i < rank; ++i) std::swap(res.perm[i], res.perm[hp[i]]);
    }
    return MODP_OK;
}

int elim_run(modp_ctx *ctx, int mode, int form, int kind, int64_t m, int64_t n, const void *A, int64_t lda,
             void *U, int64_t ldu, void *L, int64_t ldl, int64_t p, ElimResult &res)
{
    bool lost = false;
    MODP_TRY(elim_attempt(ctx, mode, form, kind, m, n, A, lda, U, ldu, L, ldl, p, res, true, &lost));
    if (!lost) return MODP_OK;
    return elim_attempt(ctx, mode, form, kind, m, n, A, lda, U, ldu, L, ldl, p, res, false, &lost);
}

// Inverse under a prime modulus: [A | I] to [U | Y] with any pivots, then
// A^{-1} = U^{-1} Y.  U is unit upper triangular, and no row order has to be undone.
int elim_inverse(modp_ctx *ctx, int form, int kind, int64_t n, const void *A, int64_t lda, void *Ainv, int64_t ldai,
                 int64_t p, int *invertible, int *taken)
{
    const ModP mp = make_modp(p);
    int st = MODP_OK;
    inverse_table(ctx, mp, &st);
    if (st != MODP_OK || !ctx->invtab_prime) return st;
    *taken = 1;
    ElimResult r;
    MODP_TRY(elim_run(ctx, ELIM_INVERSE, form, kind, n, n, A, lda, nullptr, 0, nullptr, 0, p, r));
    if (r.rank < n) return MODP_OK;
    *invertible = 1;
    const int64_t ld = rup(n, 64);
    int32_t *W = (int32_t *)ws_get(ctx, WS_WORK, sizeof(int32_t) * (size_t)ld * (size_t)(2 * n), &st);
    if (!W) return st;
    int32_t *X = (int32_t *)ws_get(ctx, WS_TRI_X, sizeof(int32_t) * (size_t)ld * (size_t)n, &st);
    if (!X) return st;
    MODP_TRY(trinv_i32(ctx, true, W, ld, X, ld, n, mp, true));
    GemmArgs g;
    g.m = n; g.n = n; g.k = n;
    g.A = X; g.lda = ld; g.ka = EK_I32;
    g.B = W + n * ld; g.ldb = ld; g.kb = EK_I32;
    g.C = Ainv; g.ldc = ldai; g.kc = kind;
    g.epi = EPI_STORE;
    g.mp = mp;
    return gemm_run(ctx, g, gemm_default_config(ctx, g, form));
}

// U of a factored W: unit upper triangular in the pivots' columns
struct Echelon {
    const int32_t *W;
    int64_t ldw, rank, nfree;
    const int32_t *pivcol, *free_cols;
    bool first;  // the pivots are in the first columns
};

static GemmArgs i32_product(int64_t m, int64_t n, int64_t k, const int32_t *A, int64_t lda, const int32_t *B, int64_t ldb,
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

// Z = U_piv^{-1} U_free (leading dimension rank rounded up to 64) by one triangular inverse and one product
static int rref_free(modp_ctx *ctx, int form, const Echelon &u, const ModP &mp, int32_t **Zout)
{
    const int64_t rank = u.rank, nfree = u.nfree, ld = rup(rank, 64);
    int st = MODP_OK;
    // pivots in the first columns: U_piv and U_free are where they are
    const int32_t *T = u.W, *Y = u.W + rank * u.ldw;
    int64_t ldt = u.ldw, ldy = u.ldw;
    if (!u.first) {
        int32_t *Tg = (int32_t *)ws_get(ctx, WS_TRI_T, sizeof(int32_t) * (size_t)ld * (size_t)rank, &st);
        if (!Tg) return st;
        int32_t *Yg = (int32_t *)ws_get(ctx, WS_INV_U, sizeof(int32_t) * (size_t)ld * (size_t)nfree, &st);
        if (!Yg) return st;
        k_gather_cols<<<grid_for(rank * rank), 256, 0, ctx->stream>>>(u.W, u.ldw, rank, u.pivcol, u.pivcol, rank, Tg, ld);
        HIP_TRY(ctx, hipGetLastError());
        k_gather_cols<<<grid_for(rank * nfree), 256, 0, ctx->stream>>>(u.W, u.ldw, rank, u.pivcol, u.free_cols, nfree, Yg, ld);
        HIP_TRY(ctx, hipGetLastError());
        T = Tg; Y = Yg;
        ldt = ldy = ld;
    }
    int32_t *X = (int32_t *)ws_get(ctx, WS_TRI_X, sizeof(int32_t) * (size_t)ld * (size_t)rank, &st);
    if (!X) return st;
    int32_t *Z = (int32_t *)ws_get(ctx, WS_INV_L, sizeof(int32_t) * (size_t)ld * (size_t)nfree, &st);
    if (!Z) return st;
    MODP_TRY(trinv_i32(ctx, true, T, ldt, X, ld, rank, mp, true));
    const GemmArgs g = i32_product(rank, nfree, rank, X, ld, Y, ldy, Z, ld, EPI_STORE, mp);
    MODP_TRY(gemm_run(ctx, g, gemm_default_config(ctx, g, form)));
    *Zout = Z;
    return MODP_OK;
}

// The same by back substitution, RB_ROWS pivots at a time and RB_COLS free
// columns at a time, written out as they are done: workspaces of about 2 RB_ROWS
// + RB_COLS columns, where the inverse and the product above take up to 2.5
// rank + 2 nfree columns and the product's residue planes.  For matrices with
// no room for those beside them: mod 65521 a whole call of 16,384^2 and rank
// 12,000 takes 46 ms instead of 44, 4096^2 and rank 3000 4.13 instead of 3.73.
constexpr int64_t RB_ROWS = 512, RB_COLS = 1024;
template <typename T>
static int rref_free_blocks(modp_ctx *ctx, int form, const Echelon &u, const ModP &mp, int64_t m, T *R, int64_t ldr)
{
    const int64_t rank = u.rank, ld = rup(rank, 64), nc = std::min(u.nfree, RB_COLS);
    int st = MODP_OK;
    int32_t *P = (int32_t *)ws_get(ctx, WS_TRI_T, sizeof(int32_t) * (size_t)ld * (size_t)RB_ROWS, &st);
    if (!P) return st;
    int32_t *X = (int32_t *)ws_get(ctx, WS_TRI_X, sizeof(int32_t) * (size_t)RB_ROWS * (size_t)rank, &st);
    if (!X) return st;
    int32_t *Y = (int32_t *)ws_get(ctx, WS_INV_U, sizeof(int32_t) * (size_t)ld * (size_t)nc, &st);
    if (!Y) return st;
    int32_t *Z = (int32_t *)ws_get(ctx, WS_INV_L, sizeof(int32_t) * (size_t)RB_ROWS * (size_t)nc, &st);
    if (!Z) return st;
    auto product = [&](const GemmArgs &g) -> int {
        const int use = form != MODP_FORM_AUTO ? form : choose_form(g.m, g.n, g.k, mp.p);
        return use == MODP_FORM_LIMB_I8 ? gemm_limb_i8(ctx, g) : gemm_plain_f64(ctx, g);
    };
    // rows [r0, r0 + rows) of the pivots' columns [c0, c0 + cols)
    auto gather = [&](int64_t r0, int64_t rows, int64_t c0, int64_t cols) -> int {
        k_gather_cols<<<grid_for(rows * cols), 256, 0, ctx->stream>>>(u.W + r0, u.ldw, rows, u.pivcol + r0,
                                                                      u.pivcol + c0, cols, P, ld);
        return hip_check(ctx, hipGetLastError(), "k_gather_cols launch");
    };
    const int64_t blocks = (rank + RB_ROWS - 1) / RB_ROWS;
    for (int64_t b = 0; b < blocks; ++b) {
        const int64_t r0 = b * RB_ROWS, nb = std::min(RB_ROWS, rank - r0);
        MODP_TRY(gather(r0, nb, r0, nb));
        MODP_TRY(trinv_i32(ctx, true, P, ld, X + r0 * RB_ROWS, RB_ROWS, nb, mp, true));
    }
    for (int64_t f0 = 0; f0 < u.nfree; f0 += nc) {
        const int64_t nf = std::min(nc, u.nfree - f0);
        k_gather_cols<<<grid_for(rank * nf), 256, 0, ctx->stream>>>(u.W, u.ldw, rank, u.pivcol, u.free_cols + f0, nf, Y, ld);
        HIP_TRY(ctx, hipGetLastError());
        for (int64_t b = blocks - 1; b >= 0; --b) {
            const int64_t r0 = b * RB_ROWS, nb = std::min(RB_ROWS, rank - r0);
            MODP_TRY(product(i32_product(nb, nf, nb, X + r0 * RB_ROWS, RB_ROWS, Y + r0, ld, Z, RB_ROWS, EPI_STORE, mp)));
            HIP_TRY(ctx, hipMemcpy2DAsync(Y + r0, sizeof(int32_t) * (size_t)ld, Z, sizeof(int32_t) * (size_t)RB_ROWS,
                                          sizeof(int32_t) * (size_t)nb, (size_t)nf, hipMemcpyDeviceToDevice, ctx->stream));
            if (r0 == 0) break;
            if (!u.first) MODP_TRY(gather(0, r0, r0, nb));
            MODP_TRY(product(i32_product(r0, nf, nb, u.first ? u.W + r0 * u.ldw : P, u.first ? u.ldw : ld, Z, RB_ROWS, Y,
                                         ld, EPI_SUB, mp)));
        }
        k_write_free<T><<<grid_for(m * nf), 256, 0, ctx->stream>>>(m, nf, (int)rank, u.free_cols + f0, Y, ld, R, ldr);
        HIP_TRY(ctx, hipGetLastError());
    }
    return MODP_OK;
}

// Reduced echelon form: PLE to U, unit upper triangular in the pivots' columns,
// then U_piv^{-1} U_free for the others alone (nothing at all for a matrix of
// full column rank).  Back substitution in blocks of 64 rows over every column,
// five launches a block, took 1.0 ms more: 4096^2 of rank 3000 mod 65521 5.12 ->
// 4.09 ms.
int elim_rref(modp_ctx *ctx, int form, int kind, int64_t m, int64_t n, const void *A, int64_t lda, void *R,
              int64_t ldr, int64_t p, ElimResult &res)
{
    // factor (PLE) into W without extracting L
    MODP_TRY(elim_run(ctx, ELIM_RREF, form, kind, m, n, A, lda, nullptr, 0, nullptr, 0, p, res));
    if (m <= 0 || n <= 0) return MODP_OK;
    const ModP mp = make_modp(p);
    const int64_t rank = res.rank, nfree = n - rank;
    int st = MODP_OK;
    const int64_t ldw = rup(m, 64);
    int32_t *W = (int32_t *)ws_get(ctx, WS_WORK, sizeof(int32_t) * (size_t)ldw * (size_t)n, &st);
    if (!W) return st;
    const int64_t mn = m < n ? m : n;
    const size_t npv = (size_t)mn + 64;
    int32_t *piv = (int32_t *)ws_get(ctx, WS_PIV, sizeof(int32_t) * 4 * npv, &st);
    if (!piv) return st;
    const int32_t *pivcol = piv + 3 * npv;
    int32_t *kinds = (int32_t *)ws_get(ctx, WS_SCRATCH, sizeof(int32_t) * 2 * (size_t)n, &st);
    if (!kinds) return st;
    int32_t *free_cols = kinds + n;
    k_column_kinds<<<(unsigned)((n + 255) / 256), 256, 0, ctx->stream>>>(pivcol, (int)rank, (int)n, kinds, free_cols);
    HIP_TRY(ctx, hipGetLastError());
    int32_t *Z = nullptr;
    bool blocks = false;  // where U_piv^{-1} U_free has no room (MODP_RREF_BLOCKS=1: always)
    if (rank > 0 && nfree > 0) {
        const Echelon u{W, ldw, rank, nfree, pivcol, free_cols, res.pivcols[(size_t)rank - 1] == rank};
        const char *benv = getenv("MODP_RREF_BLOCKS");
        blocks = benv && atoi(benv) != 0;
        if (!blocks) {
            st = rref_free(ctx, form, u, mp, &Z);
            if (st == MODP_ERR_OOM) {
                blocks = true;
                ctx->last_error.clear();
                for (int slot : {WS_TRI_T, WS_TRI_X, WS_TRI_TMP, WS_INV_U, WS_INV_L, WS_ALIMB, WS_BLIMB, WS_SLICES})
                    ws_drop(ctx, slot);
            } else {
                MODP_TRY(st);
            }
        }
        if (blocks)
            MODP_TRY(kind == EK_F64 ? rref_free_blocks<double>(ctx, form, u, mp, m, (double *)R, ldr)
                                    : rref_free_blocks<float>(ctx, form, u, mp, m, (float *)R, ldr));
    }
    const unsigned grid = grid_for(m * n);
    const int64_t ld = rup(rank, 64);
    if (kind == EK_F64)
        k_write_rref<double><<<grid, 256, 0, ctx->stream>>>(m, n, (int)rank, kinds, blocks, Z, ld, (double *)R, ldr);
    else
        k_write_rref<float><<<grid, 256, 0, ctx->stream>>>(m, n, (int)rank, kinds, blocks, Z, ld, (float *)R, ldr);
    HIP_TRY(ctx, hipGetLastError());
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return MODP_OK;
}
