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
//                columns are staged.  Above 16,384 rows k_panel_g does the
//                same with the panel left in W (any row count).
//     k_update   the block's other columns: the row map, and right of the
//                panel the triangular solve with L11 (rows of U) and the
//                rank-w update of every row below the pivots.
//   after the outer block: k_block_finish applies the block's row maps and
//   the solve with the block's L11 to the far columns, then one GEMM with
//   K = NBO (limb or plain form) updates the far trailing block.
#include <stdlib.h>

#include <type_traits>

#include "elim_panel.h"

namespace {

constexpr int NBO = 128;  // outer block width (K of the trailing GEMM)

// Panel factorisation for any number of rows (the register panel holds at
// most 16,384 and its keys 2^15 positions): the same outputs as k_panel from one 1024-thread workgroup that keeps the panel in
// W.  Thread t owns local rows t + 1024 q and is the only thread that reads
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
                                                 int32_t *__restrict__ grow)
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
    __shared__ uint32_t s_mv[2 * NBW][NBW];
    __shared__ int s_cnt;

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
    }
    if (tid == 0) {
        ctl->npiv = pc;
        ctl->status = status;
        ctl->ncols = consumed;
        ctl->nmap = nmap_all;
        ctl->kr0 = kr0;
        if (cursor) *cursor = kr0 + pc;
        if (abort && status != 0) *abort = 1;
    }
}

// After panel (kr0, c0, w) of the outer block [KC, FAR), in one launch:
// the panel's row moves for every other column of the block, and for the
// columns right of the panel the triangular solve with L11 (their rows of U)
// and the rank-npiv update of every row below the pivots.  The old values
// of moved rows come from the stage the panel kernel filled before anything
// moved, so no block reads a row that another block writes.  Grid: x =
// 64-row tiles from kr0 down, y = 8-column groups, the groups left of the
// panel first (moves only, done by the blocks of the first row tile).
// LAZY (p < 2^16): at most 32 products below 2^32 are summed exactly in FP64
// before one reduction; otherwise every product is reduced.
constexpr int UT_R = 64, UT_C = 8;
template <int WMAX, bool LAZY>
__global__ __launch_bounds__(256) void k_update(int32_t *__restrict__ W, int64_t ldw, int m, int KC, int FAR,
                                                int c0, int w, const PanelCtl *__restrict__ ctl,
                                                const int32_t *__restrict__ pivinv,
                                                const int32_t *__restrict__ pivcol,
                                                const int32_t *__restrict__ map_dst,
                                                const int32_t *__restrict__ stage, ModP mp,
                                                const int *__restrict__ skip)
{
    // the skip flag and the panel's counts are read together
    const int skipped = skip ? *skip : 0;
    const int npiv = ctl->npiv, nmap = ctl->nmap, kr0 = ctl->kr0;
    if (skipped || nmap == 0) return;
    constexpr int CPT = UT_C / 4;            // columns per thread
    __shared__ uint32_t Lf[WMAX][WMAX + 1];  // the panel's top w x w block
    __shared__ uint32_t Ls[WMAX][WMAX + 1];  // L11 (row i, pivot j < i)
    __shared__ uint32_t invs[WMAX];
    __shared__ int s_pj[WMAX];              // panel column of pivot i
    __shared__ int s_dst[64];               // row-map destinations
    __shared__ double Ut[UT_C][WMAX];        // U by column, then panel column (0: no pivot)
    __shared__ int s_e[UT_R];               // tile row -> row-map entry, or -1
    const int tid = threadIdx.x, cl = tid >> 6;
    const int nl = c0 - KC, nr = FAR - (c0 + w);
    const int gl = (nl + UT_C - 1) / UT_C;
    const int g = blockIdx.y;
    if (g < gl) {
        // left of the panel: the row moves only
        if (blockIdx.x != 0) return;
        const int cb = g * UT_C, nc = min(UT_C, nl - cb);
        for (int idx = tid; idx < nmap * nc; idx += 256) {
            const int e = idx % nmap, ci = cb + idx / nmap;
            W[(int64_t)map_dst[e] + (int64_t)(KC + ci) * ldw] = stage[e + 64 * ci];
        }
        return;
    }
    const int cb = (g - gl) * UT_C, nc = min(UT_C, nr - cb);
    const int ci0 = nl + cb;        // stage column of the group's first column
    const int cfirst = c0 + w + cb;  // its column in W
    const int64_t r0 = (int64_t)kr0 + (int64_t)blockIdx.x * UT_R;
    if (r0 >= m) return;  // the grid covers the most rows the panel can have
    const int64_t r = r0 + (tid & 63);
    const bool row_ok = r < m;

    // every global load is issued before anything waits for one: the
    // panel's top block, pivot columns and inverses, the row map, the
    // solve's inputs (thread k < nc: column k of the pivot rows' old
    // values), this thread's row of L and its old values.  Indices are
    // clamped into range so that the loads are unconditional; values that
    // are not needed are masked when they are used.
    constexpr int FPT = (WMAX * WMAX + 255) / 256;
    const int wl = w - 1;
    const int64_t rr = row_ok ? r : (int64_t)kr0;
    int32_t lf[FPT];
#pragma unroll
    for (int k = 0; k < FPT; ++k) {
        const int idx = tid + 256 * k, i = min(idx / WMAX, wl), jj = min(idx % WMAX, wl);
        lf[k] = W[(int64_t)(kr0 + i) + (int64_t)(c0 + jj) * ldw];
    }
    const int tw = min(tid, WMAX - 1);
    const int32_t iv = pivinv[kr0 + tw];
    const int32_t pjv = pivcol[kr0 + tw];
    const int32_t mdv = map_dst[min(tid, 63)];
    int32_t xs0[WMAX];
    const int64_t xcol = 64 * (int64_t)(ci0 + min(tid, nc - 1));
#pragma unroll
    for (int i = 0; i < WMAX; ++i) xs0[i] = stage[min(i, wl) + xcol];
    int32_t lr0[WMAX];
#pragma unroll
    for (int jj = 0; jj < WMAX; ++jj) lr0[jj] = W[rr + (int64_t)(c0 + min(jj, wl)) * ldw];
    int32_t cv[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) cv[k] = W[rr + (int64_t)(cfirst + min(cl + 4 * k, nc - 1)) * ldw];
    for (int idx = tid; idx < WMAX * UT_C; idx += 256) Ut[idx / WMAX][idx % WMAX] = 0.0;
    if (tid < UT_R) s_e[tid] = -1;
#pragma unroll
    for (int k = 0; k < FPT; ++k) {
        const int idx = tid + 256 * k;
        if (idx < WMAX * WMAX) Lf[idx / WMAX][idx % WMAX] = (idx / WMAX < w && idx % WMAX < w) ? (uint32_t)lf[k] : 0u;
    }
    if (tid < WMAX) {
        invs[tid] = (uint32_t)iv;
        s_pj[tid] = pjv - c0;
    }
    if (tid < 64) s_dst[tid] = mdv;
    uint32_t xs[WMAX];
#pragma unroll
    for (int i = 0; i < WMAX; ++i) xs[i] = i < w ? (uint32_t)xs0[i] : 0u;
    double Lr[WMAX];
#pragma unroll
    for (int jj = 0; jj < WMAX; ++jj) Lr[jj] = jj < w ? (double)lr0[jj] : 0.0;
    __syncthreads();
    if (tid >= npiv && tid < nmap) {
        const int64_t d = (int64_t)s_dst[tid] - r0;
        if (d >= 0 && d < UT_R) s_e[d] = tid;
    }
    for (int idx = tid; idx < WMAX * WMAX; idx += 256) {
        const int i = idx / WMAX, j = idx % WMAX;
        Ls[i][j] = (j < i && i < npiv) ? Lf[i][s_pj[j]] : 0u;
    }
    __syncthreads();
    // rows of U for the group's columns: thread k solves column k, right
    // looking (each solved value is subtracted from the rows below at once,
    // so the dependent chain per row is one normalisation and one FMA)
    if (tid < nc) {
        double a[WMAX];
#pragma unroll
        for (int i = 0; i < WMAX; ++i) a[i] = (double)xs[i];
#pragma unroll
        for (int j = 0; j < WMAX; ++j) {
            if (j < npiv) {
                // x_j = a_j / pivot_j mod p; for small p in FP64 throughout
                // (the reduced a_j times the inverse is below 2^32)
                const double x = LAZY ? dmod_near(dmod_near(a[j], mp) * (double)invs[j], mp)
                                      : (double)mulmod((uint32_t)a[j], invs[j], mp);
                Ut[tid][s_pj[j]] = x;
#pragma unroll
                for (int i = j + 1; i < WMAX; ++i) {
                    a[i] = fma(-(double)Ls[i][j], x, a[i]);
                    if (!LAZY) a[i] = dmod(a[i], mp);
                }
            }
        }
    }
    __syncthreads();
    if (!row_ok) return;
    const int rel = (int)(r - kr0);
    if (rel < npiv) {
        // pivot row: its row of U
        const int pj = s_pj[rel];
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int col = cl + 4 * k;
            if (col < nc) W[r + (int64_t)(cfirst + col) * ldw] = (int32_t)(uint32_t)Ut[col][pj];
        }
        return;
    }
    const int e = s_e[tid & 63];
    if (e >= 0) {
        // a row that moved here: its old values are in the stage
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int col = cl + 4 * k;
            if (col < nc) cv[k] = stage[e + 64 * (ci0 + col)];
        }
    }
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        const int col = cl + 4 * k;
        if (col < nc) {
            double acc = (double)cv[k];
#pragma unroll
            for (int jj = 0; jj < WMAX; ++jj) {
                acc = fma(-Lr[jj], Ut[col][jj], acc);
                if (!LAZY) acc = dmod(acc, mp);
            }
            W[r + (int64_t)(cfirst + col) * ldw] = (int32_t)(uint32_t)(LAZY ? dmod_near(acc, mp) : acc);
        }
    }
}

constexpr int MAXPAN = 64;  // inner panels per outer block (NBO / smallest panel width, 2)

// End of an outer block with P pivots (rows [KR, KR+P)), whose inner panels
// left their row gather maps in bmap_*: one wave per column outside the block
// [KC, FAR).  Columns left of the block get the swaps; far columns get the
// swaps, then the solve with the block's L11 (P x P, in LDS; lanes hold rows
// i and i+64), and their U rows go to Ubig (rows 0..consumed-1 indexed by
// block column, zero for block columns without a pivot).
template <bool LAZY>
__global__ __launch_bounds__(1024) void k_block_finish(int32_t *__restrict__ W, int64_t ldw, int64_t n, int KR,
                                                       int KC, int FAR, int P, int consumed, int npanels,
                                                       const int32_t *__restrict__ bmap_dst,
                                                       const int32_t *__restrict__ bmap_src,
                                                       const PanelCtl *__restrict__ bctl,
                                                       const int32_t *__restrict__ pivinv,
                                                       const int32_t *__restrict__ pivcol,
                                                       int32_t *__restrict__ Ubig, int64_t ldub, ModP mp,
                                                       const int *__restrict__ skip)
{
    if (skip && *skip) return;
    __shared__ uint32_t Ls[128][129];
    __shared__ uint32_t invs[128];
    __shared__ int ucolmap[128];
    __shared__ int s_pc[128];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < 128) {
        const int t = min(tid, P - 1);
        s_pc[tid] = pivcol[KR + t];
        invs[tid] = (uint32_t)pivinv[KR + t];
        ucolmap[tid] = -1;
    }
    __syncthreads();
    // L11 into LDS: lanes take consecutive rows of one pivot column, and
    // every load is issued before the first LDS store
    {
        constexpr int LPT = 128 * 128 / 1024;
        uint32_t lv[LPT];
#pragma unroll
        for (int k = 0; k < LPT; ++k) {
            const int idx = tid + 1024 * k, i = min(idx % 128, P - 1), j = min(idx / 128, P - 1);
            lv[k] = (uint32_t)W[(int64_t)(KR + i) + (int64_t)s_pc[j] * ldw];
        }
        // rows scaled by their pivot's inverse: the system becomes unit
        // lower triangular, so the substitution needs no multiply per step
#pragma unroll
        for (int k = 0; k < LPT; ++k) {
            const int idx = tid + 1024 * k, i = idx % 128, j = idx / 128;
            Ls[i][j] = (j < i && i < P) ? mulmod(lv[k], invs[i], mp) : 0u;
        }
    }
    if (tid < P) ucolmap[s_pc[tid] - KC] = tid;
    __syncthreads();
    const int64_t nout = n - (FAR - KC);
    const int um0 = lane < consumed ? ucolmap[lane] : -1;
    const int um1 = lane + 64 < consumed ? ucolmap[lane + 64] : -1;
    for (int64_t ci = (int64_t)blockIdx.x * 16 + wave; ci < nout; ci += (int64_t)gridDim.x * 16) {
        int64_t c = ci < KC ? ci : ci + (FAR - KC);
        int32_t *col = W + c * ldw;
        for (int t = 0; t < npanels; ++t) {
            const int nm = bctl[t].nmap;
            const int32_t *md = bmap_dst + t * 64, *ms = bmap_src + t * 64;
            uint32_t v = 0;
            int d = 0;
            if (lane < nm) { v = (uint32_t)col[ms[lane]]; d = md[lane]; }
            if (lane < nm) col[d] = (int32_t)v;
            __threadfence_block();
        }
        if (c < KC) continue;
        // forward substitution with the unit triangular system (rows and
        // right-hand side scaled by the pivots' inverses), lanes hold rows
        // lane and lane + 64: at step j every lane reduces its own sum (only
        // lane j's is used), readlane broadcasts it, and the rows below
        // subtract L[i][j] x_j.  LAZY (p < 2^16): the sums of at most 127
        // products below 2^32 stay exact in FP64 and are reduced once.
        double a0 = lane < P ? (double)mulmod((uint32_t)col[KR + lane], invs[lane], mp) : 0.0;
        double a1 = lane + 64 < P ? (double)mulmod((uint32_t)col[KR + lane + 64], invs[lane + 64], mp) : 0.0;
        for (int j = 0; j < P; ++j) {
            const double aj = j < 64 ? a0 : a1;
            const uint32_t xl = (uint32_t)(LAZY ? dmod_near(aj, mp) : aj);
            const uint32_t xj = (uint32_t)__builtin_amdgcn_readlane((int)xl, j & 63);
            const double xd = (double)xj;
            if (j < 64) {
                a0 = lane == j ? xd : a0;
                if (lane > j) {
                    a0 = fma(-(double)Ls[lane][j], xd, a0);
                    if (!LAZY) a0 = dmod(a0, mp);
                }
            } else if (lane == j - 64) {
                a1 = xd;
            }
            if (lane + 64 > j) {
                a1 = fma(-(double)Ls[lane + 64][j], xd, a1);
                if (!LAZY) a1 = dmod(a1, mp);
            }
        }
        const uint32_t x0 = (uint32_t)a0, x1 = (uint32_t)a1;
        if (lane < P) col[KR + lane] = (int32_t)x0;
        if (lane + 64 < P) col[KR + lane + 64] = (int32_t)x1;
        // Ubig rows 0..consumed-1 of this column: pivot i's value or zero
        int32_t *ucol = Ubig + (c - KC) * ldub;
        const int a0i = um0 < 0 ? 0 : um0, a1i = um1 < 0 ? 0 : um1;
        const uint32_t y00 = (uint32_t)__shfl((int)x0, a0i & 63), y01 = (uint32_t)__shfl((int)x1, a0i & 63);
        const uint32_t y10 = (uint32_t)__shfl((int)x0, a1i & 63), y11 = (uint32_t)__shfl((int)x1, a1i & 63);
        if (lane < consumed) ucol[lane] = um0 < 0 ? 0 : (int32_t)(a0i < 64 ? y00 : y01);
        if (lane + 64 < consumed) ucol[lane + 64] = um1 < 0 ? 0 : (int32_t)(a1i < 64 ? y10 : y11);
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

// clear the multipliers kept below the pivots: W[r, pivcol[j]] = 0 for r > j
__global__ void k_zero_lower(int32_t *__restrict__ W, int64_t ldw, int64_t m, int rank,
                             const int32_t *__restrict__ pivcol)
{
    const int64_t total = m * rank;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % m, j = e / m;
        if (r > j) W[r + (int64_t)pivcol[j] * ldw] = 0;
    }
}

// G[i, j] = W[r0 + i, pivcol[p0 + j]] for i < rows, j < nb
__global__ void k_gather_cols(const int32_t *__restrict__ W, int64_t ldw, int64_t r0, int64_t rows,
                              const int32_t *__restrict__ pivcol, int p0, int nb, int32_t *__restrict__ G,
                              int64_t ldg)
{
    const int64_t total = rows * nb;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = e % rows, j = e / rows;
        G[i + j * ldg] = W[r0 + i + (int64_t)pivcol[p0 + j] * ldw];
    }
}

// Back substitution with a unit upper triangular T (nb x nb, gathered into
// G) on rows [i0, i0+nb) of columns [cs, n): one wave per column.
__global__ __launch_bounds__(256) void k_trsm_upper_unit(int32_t *__restrict__ W, int64_t ldw, int64_t n, int i0,
                                                         int nb, int64_t cs, const int32_t *__restrict__ G,
                                                         int64_t ldg, ModP mp)
{
    __shared__ uint32_t Ts[64][65];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    {
        // every load issued before the first LDS store
        constexpr int TPT = 64 * 64 / 256;
        int32_t tv[TPT];
#pragma unroll
        for (int k = 0; k < TPT; ++k) {
            const int idx = tid + 256 * k, i = min(idx % 64, nb - 1), j = min(idx / 64, nb - 1);
            tv[k] = G[i + j * ldg];
        }
#pragma unroll
        for (int k = 0; k < TPT; ++k) {
            const int idx = tid + 256 * k, i = idx % 64, j = idx / 64;
            Ts[i][j] = (i < nb && j < nb) ? (uint32_t)tv[k] : 0u;
        }
    }
    __syncthreads();
    for (int64_t c = cs + (int64_t)blockIdx.x * 4 + wave; c < n; c += (int64_t)gridDim.x * 4) {
        int32_t *col = W + c * ldw + i0;
        uint32_t x = lane < nb ? (uint32_t)col[lane] : 0u;
        for (int j = nb - 1; j > 0; --j) {
            const uint32_t xj = (uint32_t)__builtin_amdgcn_readlane((int)x, j);
            if (lane < j) x = submod(x, mulmod(Ts[lane][j], xj, mp), mp);
        }
        if (lane < nb) col[lane] = (int32_t)x;
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

__global__ void k_set_int(int *p, int v) { *p = v; }

// t[a] = a^{-1} mod p for a < n, 0 where there is none
__global__ void k_inv_table(uint32_t *__restrict__ t, int n, ModP mp)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < n) t[a] = a > 0 && a < mp.p ? modinv((uint32_t)a, mp) : 0u;
}

// Inverses of the residues below PINV, from which the panels make every other
// inverse; built once per modulus and kept in the context.
const uint32_t *inverse_table(modp_ctx *ctx, const ModP &mp, int *st)
{
    if (ctx->invtab && ctx->invtab_p == mp.p) return ctx->invtab;
    if (!ctx->invtab) {
        hipError_t e = hipMalloc(&ctx->invtab, sizeof(uint32_t) * PINV);
        if (e != hipSuccess) { *st = hip_check(ctx, e, "inverse table"); return nullptr; }
    }
    k_inv_table<<<PINV / 256, 256, 0, ctx->stream>>>(ctx->invtab, PINV, mp);
    if (hipGetLastError() != hipSuccess) { *st = MODP_ERR_DEVICE; return nullptr; }
    ctx->invtab_p = mp.p;
    return ctx->invtab;
}

}  // namespace

int elim_run(modp_ctx *ctx, int mode, int form, int kind, int64_t m, int64_t n, const void *A, int64_t lda,
             void *U, int64_t ldu, void *L, int64_t ldl, int64_t p, ElimResult &res)
{
    const ModP mp = make_modp(p);
    const bool ple = mode != ELIM_PLUQ;
    const int64_t mn = m < n ? m : n;
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
    // W-resident panel beyond 16,384 rows.  Mod 65521 a 32-column panel takes
    // 37 us on one workgroup and 49 us on an XCD, whatever its rows (one
    // workgroup with 512 rows, two waves per SIMD: 58 us).
    // MODP_PANEL_GLOBAL=1 sends every panel to the W-resident kernel (used
    // to compare the two panel kernels at sizes both handle)
    const char *genv = getenv("MODP_PANEL_GLOBAL");
    const bool force_global = genv && atoi(genv) != 0;
    // the cycles that a workgroup of a panel on one XCD waits for the others to
    // start before the panel is left to the W-resident kernel
    // (MODP_PANEL_PATIENCE sets it: 0 makes every such panel give up)
    const char *penv = getenv("MODP_PANEL_PATIENCE");
    const long long patience = penv ? atoll(penv) : 50000000LL;
    bool gave_up = false;  // in the previous outer block
    auto panel_width = [&](int64_t KR) {
        return force_global || gave_up || m - KR > PMULTI ? GNBW : PNW;
    };

    int st = MODP_OK;
    const int64_t ldw = rup(m, 64);
    int32_t *W = (int32_t *)ws_get(ctx, WS_WORK, sizeof(int32_t) * (size_t)ldw * (size_t)n, &st);
    if (!W) return st;
    // pivot arrays, per-panel control blocks and row gather maps of one outer block
    const size_t npv = (size_t)mn + 64;
    const size_t piv_bytes = sizeof(int32_t) * (4 * npv + 2 * MAXPAN * 64) + sizeof(PanelCtl) * MAXPAN + 512 +
                             sizeof(int32_t) * 64 * NBO;
    int32_t *piv = (int32_t *)ws_get(ctx, WS_PIV, piv_bytes, &st);
    if (!piv) return st;
    int32_t *ipiv = piv, *pivval = piv + npv, *pivinv = piv + 2 * npv, *pivcol = piv + 3 * npv;
    int32_t *bmap_dst = piv + 4 * npv, *bmap_src = bmap_dst + MAXPAN * 64;
    PanelCtl *bctl = (PanelCtl *)(bmap_src + MAXPAN * 64);
    int *flag = (int *)(bctl + MAXPAN);
    int *abort_flag = flag + 1;
    int *cursor = flag + 2;                         // first row of the next panel (lu, rref)
    uint32_t *arrive = (uint32_t *)(flag + 4);      // one word per panel of the block
    int32_t *stage = (int32_t *)(arrive + MAXPAN);  // moved rows' old values, 64 x NBO
    int32_t *Ubig = (int32_t *)ws_get(ctx, WS_UBUF, sizeof(int32_t) * (size_t)NBO * (size_t)(n + 1), &st);
    if (!Ubig) return st;
    // row positions of the W-resident panel (position of each row, row at
    // each position)
    int32_t *gpos = nullptr, *grow = nullptr;
    if (force_global || m > PSINGLE) {
        gpos = (int32_t *)ws_get(ctx, WS_GPOS, sizeof(int32_t) * 2 * (size_t)m, &st);
        if (!gpos) return st;
        grow = gpos + m;
    }
    PanelCtl *hctl = (PanelCtl *)pinned_get(ctx, sizeof(PanelCtl) * (MAXPAN + 1) + 64, &st);
    if (!hctl) return st;

    MODP_TRY(util_convert(ctx, kind, m, n, A, lda, EK_I32, W, ldw, mp));
    const uint32_t *invs = inverse_table(ctx, mp, &st);
    if (st != MODP_OK) return st;
    // exchange area of the panels on one XCD: its words are recognised by
    // tags that count the context's panels, so old ones are cleared only when
    // the 17 bits of a key's tag (the 32 of a residue's) have been through
    PanelExchange *xch = nullptr;
    if (!force_global && m > PSINGLE) {
        const bool fresh = !ctx->ws[WS_PANEL];
        xch = (PanelExchange *)ws_get(ctx, WS_PANEL, sizeof(PanelExchange), &st);
        if (!xch) return st;
        if (fresh) ctx->panel_tag = 0;
    }
    auto next_tag = [&](uint32_t *t) -> int {
        if ((ctx->panel_tag & 0x1ffffu) == 0)
            HIP_TRY(ctx, hipMemsetAsync(xch, 0, ctx->panel_tag == 0 ? sizeof(PanelExchange) : sizeof(xch->key),
                                        ctx->stream));
        *t = ctx->panel_tag;
        ctx->panel_tag += 64;
        return MODP_OK;
    };

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
        if (use_form == MODP_FORM_LIMB_I8) return gemm_limb_i8(ctx, g);
        return gemm_plain_f64(ctx, g);
    };
    // panel t of the current outer block at (rj, cj), width w; it has at most
    // m - rj rows
    auto launch_panel_t = [&](int width, int t, int64_t KC, int64_t FAR, int64_t rj, int64_t cj, int64_t w, int *abort,
                              int *cursor) -> int {
        if (t >= MAXPAN) return set_error(ctx, MODP_ERR_DEVICE, "more than %d panels in an outer block", MAXPAN);
        int32_t *mdst = bmap_dst + t * 64, *msrc = bmap_src + t * 64;
        PanelCtl *pctl = bctl + t;
        TimedLaunch tl(ctx, "elim_panel");
        if (width == GNBW) {
            k_panel_g<GNBW><<<1, GPT, 0, ctx->stream>>>(W, ldw, (int)m, (int)rj, (int)cj, (int)w, mp, ple, ipiv,
                                                        pivval, pivinv, pivcol, mdst, msrc, pctl, abort,
                                                        (int)KC, (int)FAR, stage, cursor, gpos, grow);
            return hip_check(ctx, hipGetLastError(), "k_panel_g launch");
        }
        PanelArgs a = {};
        a.W = W; a.ldw = ldw; a.m = (int)m; a.kr0 = (int)rj; a.c0 = (int)cj; a.w = (int)w; a.ple = ple;
        a.KC = (int)KC; a.FAR = (int)FAR; a.mp = mp; a.invs = invs;
        a.ipiv = ipiv; a.pivval = pivval; a.pivinv = pivinv; a.pivcol = pivcol;
        a.map_dst = mdst; a.map_src = msrc; a.stage = stage; a.ctl = pctl; a.abort = abort; a.cursor = cursor;
        const int mode = mp.small ? 0 : mp.p <= ((int64_t)1 << 24) ? 1 : 2;
        if (m - rj <= PSINGLE) {
            if (mode == 0) k_panel<false, 0><<<1, PSINGLE, 0, ctx->stream>>>(a);
            else if (mode == 1) k_panel<false, 1><<<1, PSINGLE, 0, ctx->stream>>>(a);
            else k_panel<false, 2><<<1, PSINGLE, 0, ctx->stream>>>(a);
            return hip_check(ctx, hipGetLastError(), "k_panel launch");
        }
        a.x = xch;
        a.arrive = arrive + t;
        a.G = (int)((m - rj + 255) / 256);
        a.patience = patience;
        MODP_TRY(next_tag(&a.tag));
        const unsigned grid = 8 * (a.G - 1) + 1;
        if (mode == 0) k_panel<true, 0><<<grid, 256, 0, ctx->stream>>>(a);
        else if (mode == 1) k_panel<true, 1><<<grid, 256, 0, ctx->stream>>>(a);
        else k_panel<true, 2><<<grid, 256, 0, ctx->stream>>>(a);
        return hip_check(ctx, hipGetLastError(), "k_panel launch");
    };
    // abort flag, cursor and arrival words of a block
    auto block_begin = [&]() -> int {
        return hip_check(ctx, hipMemsetAsync(abort_flag, 0, (size_t)((char *)(arrive + MAXPAN) - (char *)abort_flag),
                                             ctx->stream), "block flags");
    };
    // the rest of the outer block after panel t: its row moves, and right
    // of the panel the rows of U and the rank-npiv update below the pivots
    auto update_t = [&](int t, int64_t KC, int64_t FAR, int64_t rj, int64_t cj, int64_t w, const int *skip) -> int {
        const int64_t nl = cj - KC, nr = FAR - (cj + w);
        const unsigned gy = (unsigned)((nl + UT_C - 1) / UT_C + (nr + UT_C - 1) / UT_C);
        if (gy == 0) return MODP_OK;
        const dim3 grid((unsigned)((m - rj + UT_R - 1) / UT_R), gy);
        TimedLaunch tl(ctx, "elim_update");
#define LAUNCH_UPDATE(WM_) \
    if (mp.small) \
        k_update<WM_, true><<<grid, 256, 0, ctx->stream>>>(W, ldw, (int)m, (int)KC, (int)FAR, (int)cj, (int)w, \
                                                           bctl + t, pivinv, pivcol, bmap_dst + t * 64, stage, mp, skip); \
    else \
        k_update<WM_, false><<<grid, 256, 0, ctx->stream>>>(W, ldw, (int)m, (int)KC, (int)FAR, (int)cj, (int)w, \
                                                            bctl + t, pivinv, pivcol, bmap_dst + t * 64, stage, mp, skip);
        if (w <= 8) {
            LAUNCH_UPDATE(8)
        } else if (w <= 16) {
            LAUNCH_UPDATE(16)
        } else {
            LAUNCH_UPDATE(32)
        }
#undef LAUNCH_UPDATE
        return hip_check(ctx, hipGetLastError(), "k_update launch");
    };
    // end of an outer block with P pivots over `consumed` columns
    auto block_end = [&](int64_t KR, int64_t KC, int64_t FAR, int64_t P, int64_t consumed, int npanels,
                         const int *skip) -> int {
        if (P <= 0) return MODP_OK;
        const int64_t nout = n - (FAR - KC);
        if (nout > 0) {
            TimedLaunch tl(ctx, "elim_block_finish");
            int64_t g = (nout + 15) / 16;
            if (g > 2048) g = 2048;
            if (mp.small)
                k_block_finish<true><<<(unsigned)g, 1024, 0, ctx->stream>>>(
                    W, ldw, n, (int)KR, (int)KC, (int)FAR, (int)P, (int)consumed, npanels, bmap_dst, bmap_src, bctl,
                    pivinv, pivcol, Ubig, NBO, mp, skip);
            else
                k_block_finish<false><<<(unsigned)g, 1024, 0, ctx->stream>>>(
                    W, ldw, n, (int)KR, (int)KC, (int)FAR, (int)P, (int)consumed, npanels, bmap_dst, bmap_src, bctl,
                    pivinv, pivcol, Ubig, NBO, mp, skip);
            HIP_TRY(ctx, hipGetLastError());
        }
        const int64_t rbeg = KR + P;
        return gemm_sub(rbeg, m - rbeg, FAR, n - FAR, KC, consumed, Ubig + (FAR - KC) * NBO, skip);
    };

    std::vector<int64_t> col_stack;
    int64_t kr = 0, kc = 0, last = n - 1;
    bool done = false;
    while (!done && kr < m && kc < n) {
        // ---- one outer block of columns [KC, FAR) ----
        const int64_t KR = kr, KC = kc;
        const int64_t colend = ple ? n : last + 1;  // columns usable as pivot columns
        int64_t nbo = colend - KC;
        if (nbo > NBO) nbo = NBO;
        if (nbo < 0) nbo = 0;  // pluq: only moved zero columns remain
        const int64_t FAR = KC + nbo;
        const int NBW = panel_width(KR);
        gave_up = false;
        bool stop_zero = false;
        if (!ple && nbo > 0) {
            // pluq: every panel of the block is enqueued assuming it finds a
            // pivot in each column; a panel that meets a zero column raises
            // the abort flag, which turns the rest of the block into no-ops,
            // and the block is completed from the host after one sync
            MODP_TRY(block_begin());
            std::vector<int64_t> pr, pcj, pw;
            for (int64_t cj = KC; cj < FAR;) {
                const int64_t rj = KR + (cj - KC);
                if (rj >= m) break;
                int64_t w = FAR - cj;
                if (w > NBW) w = NBW;
                if (w > m - rj) w = m - rj;
                pr.push_back(rj); pcj.push_back(cj); pw.push_back(w);
                cj += w;
            }
            const int np = (int)pr.size();
            int64_t Pfull = 0;
            for (int t = 0; t < np; ++t) {
                MODP_TRY(launch_panel_t(NBW, t, KC, FAR, pr[t], pcj[t], pw[t], abort_flag, nullptr));
                MODP_TRY(update_t(t, KC, FAR, pr[t], pcj[t], pw[t], abort_flag));
                Pfull += pw[t];
            }
            MODP_TRY(block_end(KR, KC, FAR, Pfull, Pfull, np, abort_flag));
            // the control blocks and, right after them, the flags: one copy
            HIP_TRY(ctx, hipMemcpyAsync(hctl, bctl, sizeof(PanelCtl) * MAXPAN + 2 * sizeof(int), hipMemcpyDeviceToHost,
                                        ctx->stream));
            HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
            const int aborted = reinterpret_cast<const int *>(hctl + MAXPAN)[1];
            if (!aborted) {
                kr += Pfull;
                kc += Pfull;
            } else {
                int ts = 0;
                while (ts < np && hctl[ts].status == 0) ++ts;
                if (ts >= np)
                    return set_error(ctx, MODP_ERR_DEVICE, "elimination pipeline aborted without a stopping panel");
                if (hctl[ts].status == 3)
                    return set_error(ctx, MODP_ERR_NOT_INVERTIBLE,
                                     "pivot has no inverse modulo %lld (modulus not prime)", (long long)p);
                if (hctl[ts].status == 6)
                    return set_error(ctx, MODP_ERR_DEVICE, "an elimination panel's exchange did not end");
                gave_up = hctl[ts].status == 5;
                const int64_t npiv = hctl[ts].npiv;
                int64_t P = 0;
                for (int t = 0; t < ts; ++t) P += pw[t];
                if (npiv > 0) MODP_TRY(update_t(ts, KC, FAR, pr[ts], pcj[ts], pw[ts], nullptr));
                P += npiv;
                MODP_TRY(block_end(KR, KC, FAR, P, P, ts + 1, nullptr));
                kr += P;
                kc += P;
                stop_zero = hctl[ts].status == 1;
            }
        } else if (nbo > 0) {
            // ple: panels skip zero columns, so a panel's first row depends
            // on the pivots found before it.  The panels of the block are
            // enqueued at their fixed columns and each takes its first row
            // from a device cursor that the previous one advanced; the
            // updates read it from the panel's control block.  A panel that
            // runs out of rows (or meets a pivot without inverse) raises the
            // abort flag, which turns the rest of the block into no-ops, and
            // the host reads the outcome once per block.
            MODP_TRY(block_begin());
            k_set_int<<<1, 1, 0, ctx->stream>>>(cursor, (int)KR);
            HIP_TRY(ctx, hipGetLastError());
            std::vector<int64_t> pcj, pw;
            for (int64_t cj = KC; cj < FAR; cj += NBW) {
                pcj.push_back(cj);
                pw.push_back(std::min<int64_t>(NBW, FAR - cj));
            }
            const int np = (int)pcj.size();
            for (int t = 0; t < np; ++t) {
                MODP_TRY(launch_panel_t(NBW, t, KC, FAR, KR, pcj[t], pw[t], abort_flag, cursor));
                MODP_TRY(update_t(t, KC, FAR, KR, pcj[t], pw[t], abort_flag));
            }
            HIP_TRY(ctx, hipMemcpyAsync(hctl, bctl, sizeof(PanelCtl) * np, hipMemcpyDeviceToHost, ctx->stream));
            HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
            int64_t P = 0, consumed = 0;
            int npanels = 0;
            for (int t = 0; t < np; ++t) {
                const PanelCtl &pc = hctl[t];
                if (pc.status == 4) break;
                ++npanels;
                if (pc.status == 3)
                    return set_error(ctx, MODP_ERR_NOT_INVERTIBLE,
                                     "pivot has no inverse modulo %lld (modulus not prime)", (long long)p);
                if (pc.status == 6)
                    return set_error(ctx, MODP_ERR_DEVICE, "an elimination panel's exchange did not end");
                gave_up = pc.status == 5;
                P += pc.npiv;
                consumed += pc.ncols;
                if (pc.status != 0) {
                    // the update after this panel was skipped by its own flag
                    if (pc.npiv > 0) MODP_TRY(update_t(t, KC, FAR, KR, pcj[t], pw[t], nullptr));
                    break;
                }
            }
            kr += P;
            kc += consumed;
            MODP_TRY(block_end(KR, KC, FAR, P, consumed, npanels, nullptr));
            if (P < consumed && kr < m && kc < n) {
                // the block met zero columns: if nothing nonzero is left
                // below row kr, no later column has a pivot and the
                // factorisation is complete (rank = kr)
                HIP_TRY(ctx, hipMemsetAsync(flag, 0, sizeof(int), ctx->stream));
                k_any_nonzero<<<grid_for((m - kr) * (n - kc), 4096), 256, 0, ctx->stream>>>(W, ldw, kr, m, kc, n, flag);
                HIP_TRY(ctx, hipGetLastError());
                int *hflag = (int *)hctl;
                HIP_TRY(ctx, hipMemcpyAsync(hflag, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
                HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
                if (!*hflag) done = true;
            }
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

// Back-elimination of a PLE-reduced working array into RREF: row blocks of
// 64 pivots from the bottom; each block is first reduced in place (unit upper
// triangular solve) and then eliminated from every row above it by a GEMM.
int elim_rref(modp_ctx *ctx, int form, int kind, int64_t m, int64_t n, const void *A, int64_t lda, void *R,
              int64_t ldr, int64_t p, ElimResult &res)
{
    // factor (PLE) into W without extracting L
    MODP_TRY(elim_run(ctx, ELIM_RREF, form, kind, m, n, A, lda, nullptr, 0, nullptr, 0, p, res));
    const ModP mp = make_modp(p);
    const int64_t rank = res.rank;
    int st = MODP_OK;
    const int64_t ldw = rup(m, 64);
    int32_t *W = (int32_t *)ws_get(ctx, WS_WORK, sizeof(int32_t) * (size_t)ldw * (size_t)n, &st);
    if (!W) return st;
    const int64_t mn = m < n ? m : n;
    const size_t npv = (size_t)mn + 64;
    int32_t *piv = (int32_t *)ws_get(ctx, WS_PIV, sizeof(int32_t) * (4 * npv + 4 * 64) + sizeof(PanelCtl) + 64, &st);
    if (!piv) return st;
    int32_t *pivcol = piv + 3 * npv;
    if (rank > 0) {
        k_zero_lower<<<grid_for(m * rank), 256, 0, ctx->stream>>>(W, ldw, m, (int)rank, pivcol);
        HIP_TRY(ctx, hipGetLastError());
    }
    if (rank > 1) {
        int32_t *G = (int32_t *)ws_get(ctx, WS_SCRATCH, sizeof(int32_t) * (size_t)(rank + 64) * 64, &st);
        if (!G) return st;
        for (int64_t i1 = rank; i1 > 0;) {
            const int64_t i0 = i1 > 64 ? i1 - 64 : 0;
            const int nb = (int)(i1 - i0);
            // first pivot column of the block (the factorisation returned
            // the pivot columns, 1-based)
            const int64_t cs = res.pivcols[(size_t)i0] - 1;
            // T = W[i0:i1, pivcol[i0:i1]] -> G (nb x nb), then reduce the block
            k_gather_cols<<<grid_for((int64_t)nb * nb), 256, 0, ctx->stream>>>(W, ldw, i0, nb, pivcol, (int)i0, nb, G, 64);
            HIP_TRY(ctx, hipGetLastError());
            k_trsm_upper_unit<<<grid_for((n - cs) * 64, 4096), 256, 0, ctx->stream>>>(W, ldw, n, (int)i0, nb, cs, G, 64, mp);
            HIP_TRY(ctx, hipGetLastError());
            if (i0 > 0) {
                // M = W[0:i0, pivcol[i0:i1]] -> G (i0 x nb); W[0:i0, cs:] -= M * W[i0:i1, cs:]
                k_gather_cols<<<grid_for(i0 * nb), 256, 0, ctx->stream>>>(W, ldw, 0, i0, pivcol, (int)i0, nb, G, i0);
                HIP_TRY(ctx, hipGetLastError());
                GemmArgs g;
                g.m = i0; g.n = n - cs; g.k = nb;
                g.A = G; g.lda = i0; g.ka = EK_I32;
                g.B = W + i0 + cs * ldw; g.ldb = ldw; g.kb = EK_I32;
                g.C = W + cs * ldw; g.ldc = ldw; g.kc = EK_I32;
                g.epi = EPI_SUB;
                g.mp = mp;
                const int bform = form != MODP_FORM_AUTO ? form : choose_form(g.m, g.n, g.k, p);
                if (bform == MODP_FORM_LIMB_I8 && nb >= 64) MODP_TRY(gemm_limb_i8(ctx, g));
                else MODP_TRY(gemm_plain_f64(ctx, g));
            }
            i1 = i0;
        }
    }
    unsigned g = grid_for(m * n);
    if (kind == EK_F64) k_extract_u<double><<<g, 256, 0, ctx->stream>>>(m, n, W, ldw, (int)rank, pivcol, (double *)R, ldr);
    else k_extract_u<float><<<g, 256, 0, ctx->stream>>>(m, n, W, ldw, (int)rank, pivcol, (float *)R, ldr);
    HIP_TRY(ctx, hipGetLastError());
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return MODP_OK;
}
