/*
 * Whole-GPU multifrontal LU of one large sparse system: the replacement of
 * klu_refactor (klu_refactor.c:18-482) and klu_solve (klu_solve.c:14-400)
 * for systems far beyond one wave's LDS program, such as the 1024 x 1024
 * power-grid mesh (~1.1M unknowns).  The symbolic phase (splu_host.cpp)
 * fixes the pivot sequence and the frontal tree; this file holds the numeric
 * kernels and the C ABI.
 *
 * Refactor, by tree height, leaves first:
 *   k_sp_small    fronts of up to SPLU_SMALL unknowns, a workgroup each:
 *                 CSC entries and children's Schur complements assembled in
 *                 LDS, factored there, written once;
 *   larger fronts:
 *   k_sp_asm      assembles 16 columns a workgroup from the children's Schur
 *                 complements (by inverse index lists: each entry is written
 *                 once and never cleared first) and the CSC entries;
 *                 k_sp_asm_many a column a wavefront, of fronts of more than
 *                 SPLU_KIDS children;
 *   k_sp_panel    per 64-column panel: the diagonal block factored in LDS by
 *                 16-column steps (Doolittle, no pivoting), then L21 rows
 *                 and U12 columns by substitution, one a thread;
 *   k_sp_update   the trailing block minus L21 U12 on the matrix cores, 64 x
 *                 64 tiles.
 * Solve: rows permuted (k_sp_perm), forward substitution leaves first with
 * each front's boundary part handed to its parent, backward from the root.
 * Small fronts take a workgroup each; the larger run 64 pivots a launch,
 * every workgroup with 256 of the rows below (above).
 * Every write has one writer and a fixed order, so the results are the same
 * run to run.
 *
 * What bounds it on the 1024 x 1024 mesh (33 GFLOP, 1.2 GB of L + U: 0.46 and
 * 0.24 ms on this card): the chain of heights, 65 panels of the top fronts one
 * after the other, where 1-30 fronts leave most of the chip idle.  Factor and
 * solve 9.7 ms: panels 65 x 42 us, updates 65 x 26, small fronts 2.0 ms,
 * assembly 0.5, the solves 2.5.  With 32-column panels for every height, a
 * cleared and scattered-to store and an extend-add launch per child it was 15.8
 * ms: 250 panels and updates of 41 and 39 us, 1.25 ms of extend-adds, 0.57 of
 * clearing and scattering; on a 93 x 93 mesh 0.86 ms, now 0.63.
 */
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "ngmi_internal.h"
#include "splu_types.h"
#include "fp64.h"

using namespace ngmi;

namespace {

constexpr int WG = 256;
constexpr int NB = SPLU_NB;
constexpr int DB = 16;        /* columns a diagonal block is factored by: the lanes a DPP row broadcasts along */
constexpr int DLD = NB + 1;   /* leading dimension of a panel's diagonal block in LDS */

typedef double d4 __attribute__((ext_vector_type(4)));

/* a wave-uniform lane's double, through two scalar readlanes */
__device__ __forceinline__ double rdlane(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

/* div_by gives num / d, a positive zero's included */
__device__ __forceinline__ bool div_by_ok(double num, double d)
{
    return div_by_divisor(d) && (div_by_dividend(num) || __double_as_longlong(num) == 0);
}

/* v of lane N of each row of 16 lanes, to the row (one v_mov_b64_dpp; every
 * lane of the wave has to be active) */
template <int N>
__device__ __forceinline__ double bcast16(double v)
{
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0LL, (long long)__double_as_longlong(v), 0x150 + N, 0xf, 0xf, true));
}

/* v is formed here: left alone, the compiler puts an elimination step's
 * products off to where their sums are read, and holds every operand till
 * then */
__device__ __forceinline__ void pin(double &v) { asm volatile("" : "+v"(v)); }

/* this wavefront's number in its workgroup, as a scalar */
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

/* f(std::integral_constant<int, B>()) ... f(<E - 1>) */
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>());
        static_for<B + 1, E>(f);
    }
}

struct SpDev {
    const SpluFront *front;
    const SpluKid *kid;
    const int *idx, *ent_src, *cg, *gk, *inv, *up_ptr, *rel;
    const SpluUp *up_ent;
    const uint32_t *ent_rc;
};

__global__ void k_sp_clear(int *flag)
{
    if (threadIdx.x < 4) flag[threadIdx.x] = 0;
}

/* the largest multiplier of a workgroup's lanes into flag[2..3] (a double's
 * bits, atomic max): a pivot sequence fixed in advance has no threshold test,
 * and KLU's partial pivoting (tol 1e-3, klu_kernel.c:370-530) would have
 * exchanged any pivot whose column holds a multiplier above 1/tol.  Every
 * lane takes part. */
__device__ __forceinline__ void report_lmax(double lmax, int *flag)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lmax = fmax(lmax, __shfl_xor(lmax, o));
    if ((threadIdx.x & 63) == 0 && lmax > 0.0)
        atomicMax(reinterpret_cast<unsigned long long *>(flag + 2), (unsigned long long)__double_as_longlong(lmax));
}

/* Doolittle LU, no pivoting, of the w x w block (w <= DB) at S[c * ld + r],
 * by one whole wavefront: lane j of each row of 16 holds column j; at step k
 * every later column subtracts column k, broadcast along the lanes by DPP
 * moves, times its own row-k entry over the pivot.  inv takes the pivots'
 * reciprocals.  Returns the lane's largest multiplier; *bad: a zero or
 * non-finite pivot.  A chain of w dependent steps of ~400 cycles, each with
 * a reciprocal; through v_readlane, 32 columns wide, ~550. */
__device__ __forceinline__ double diag_lu(double *S, int ld, int w, double *inv, bool *bad_out)
{
    const int lane = threadIdx.x & 63, j = lane & (DB - 1);
    double c[DB];
    {
        const double *col = S + min(j, w - 1) * ld;
#pragma unroll
        for (int i = 0; i < DB; i++) c[i] = col[min(i, w - 1)];
    }
    double dinv = 0.0;
    bool bad = false;
    static_for<0, DB>([&](auto kc) {
        constexpr int k = kc;
        if (k < w) {
            const double piv = bcast16<k>(c[k]), iv = recip(piv);
            bad |= !(fabs(piv) > 0.0) || !isfinite(piv);
            if (j == k) dinv = iv;
            const double nu = j > k ? -(c[k] * iv) : 0.0;
            static_for<k + 1, DB>([&](auto ic) {
                c[ic] = fma(bcast16<k>(c[ic]), nu, c[ic]);
                pin(c[ic]);
            });
        }
    });
    double lmax = 0.0;
    if (lane < DB) {
        inv[j] = dinv;
        if (j < w) {
#pragma unroll
            for (int i = 0; i < DB; i++)
                if (i < w) {
                    /* column j's multipliers: below the diagonal, over its pivot */
                    if (i > j) {
                        c[i] *= dinv;
                        lmax = fmax(lmax, fabs(c[i]));
                    }
                    S[j * ld + i] = c[i];
                }
        }
    }
    *bad_out = bad;
    return lmax;
}

/* x (w entries st apart in LDS) against the factored block D (column-major,
 * ld), by a whole wavefront, a row (x U = row) or column (L x = column) a
 * lane; live: this lane's result is stored.  The block's entries are held 16
 * lanes a row and broadcast by DPP moves: read from LDS by every lane, each
 * is a 512 B broadcast, and four waves of them keep the LDS busy for longer
 * than the arithmetic takes.  Step k's are read during step k - 1.  Returns
 * the row's largest entry. */
__device__ __forceinline__ double blk_solve(double *xs, int st, int w, const double *D, int ld, const double *inv,
                                            bool row, bool live)
{
    const int j = threadIdx.x & (DB - 1);
    double x[DB], lmax = 0.0;
#pragma unroll
    for (int k = 0; k < DB; k++) x[k] = xs[min(k, w - 1) * st];
    const int jw = min(j, w - 1), ks = row ? 1 : ld, a0 = row ? jw * ld : jw;
    const double iv = inv[j];
    double u = D[a0];
    static_for<0, DB>([&](auto kc) {
        constexpr int k = kc;
        if (k < w) {
            const double m = u;
            asm volatile("" ::: "memory");
            if constexpr (k + 1 < DB) u = D[a0 + min(k + 1, w - 1) * ks];
            if (row) x[k] *= bcast16<k>(iv);
            const double nx = -x[k];
            static_for<k + 1, DB>([&](auto qc) {
                constexpr int q = qc;
                x[q] = fma(bcast16<q>(m), nx, x[q]);
                pin(x[q]);
            });
        }
    });
    if (!live) return 0.0;
#pragma unroll
    for (int k = 0; k < DB; k++)
        if (k < w) {
            xs[k * st] = x[k];
            lmax = fmax(lmax, fabs(x[k]));
        }
    return row ? lmax : 0.0;
}

/* the rows below and columns right of the w x w diagonal block at (kb, kb)
 * of S, up to index n, 64 a wave from wave wv of nw on.  Returns the lane's
 * largest multiplier. */
__device__ __forceinline__ double lds_solves(double *S, int ld, int kb, int w, int n, const double *inv,
                                             int wv, int nw)
{
    const int t0 = kb + w, m = n - t0, items = (m + 63) / 64;
    double lmax = 0.0;
    for (int it = wv; it < 2 * items; it += nw) {
        const bool row = it < items;
        const int t = (row ? it : it - items) * 64 + (int)(threadIdx.x & 63), i = t0 + min(t, m - 1);
        const double l = blk_solve(row ? S + kb * ld + i : S + i * ld + kb, row ? ld : 1, w, S + kb * ld + kb, ld,
                                   inv, row, t < m);
        lmax = fmax(lmax, l);
    }
    return lmax;
}

/* NT 16 x 16 tiles (r0[t], c0[t]) of S -= S[:, kb:kb+w] S[kb:kb+w, :] on the
 * matrix cores, side by side so that one's LDS reads cover the other's
 * products.  v_mfma_f64_16x16x4: lane l gives operand rows / columns l % 16
 * at depth l / 16 and receives rows 4 v + l / 16, column l % 16; U is the row
 * operand, so that 16 neighbouring lanes hold 16 consecutive rows of a
 * column of the result.  Indices are below 2^16: 24-bit products. */
template <int NT>
__device__ __forceinline__ void lds_tile(double *S, int ld, int kb, int w, int n, const int *r0, const int *c0)
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    double cur[NT][4];
    int at[NT][4], row[NT], ua[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        row[t] = min(r0[t] + li, n - 1);
        ua[t] = __mul24(min(c0[t] + li, n - 1), ld) + kb;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            at[t][q] = __mul24(min(c0[t] + 4 * q + lk, n - 1), ld) + row[t];
            cur[t][q] = S[at[t][q]];
        }
    }
    d4 acc[NT] = {};
    double l[NT][4], u[NT][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = min(4 * q + lk, w - 1);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            l[t][q] = S[__mul24(kb + k, ld) + row[t]];
            u[t][q] = S[ua[t] + k];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int t = 0; t < NT; t++)
            acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(4 * q + lk < w ? u[t][q] : 0.0, l[t][q], acc[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (r0[t] + li < n && c0[t] + 4 * v + lk < n) S[at[t][v]] = cur[t][v] - acc[t][v];
}

/* tiles t, t + nw, .. (t < nw) of the T x T block from t0 on, column by
 * column; positions step by nw instead of being divided out of t.  corner:
 * tile (0, 0), the next diagonal block, is another wave's. */
__device__ __forceinline__ void lds_update(double *S, int ld, int kb, int w, int n, int t, int nw, bool corner)
{
    const int t0 = kb + w, T = (n - t0 + 15) >> 4;
    int r = t, c = 0;
    auto wrap = [&]() {
        while (r >= T) r -= T, c++;
    };
    auto settle = [&]() {
        wrap();
        if (corner && r == 0 && c == 0) {
            r += nw;
            wrap();
        }
    };
    if (T > 0) settle();
    while (T > 0 && c < T) {
        int r0[2], c0[2];
        r0[0] = t0 + 16 * r;
        c0[0] = t0 + 16 * c;
        r += nw;
        settle();
        if (c < T) {
            r0[1] = t0 + 16 * r;
            c0[1] = t0 + 16 * c;
            r += nw;
            settle();
            lds_tile<2>(S, ld, kb, w, n, r0, c0);
        } else {
            lds_tile<1>(S, ld, kb, w, n, r0, c0);
        }
    }
}

/* child q's boundary index of the front's unknowns, or -1, staged in LDS */
constexpr int KID_LDS = 4;

/* One front of up to SPLU_SMALL unknowns a workgroup, in LDS with an odd
 * leading dimension (columns and rows both free of bank conflicts).  Every
 * entry is gathered from the children by inverse index lists: nothing is
 * cleared, and the children's loads do not wait for one another as they do
 * when one after the other is added through its own index list. */
template <int T>
__global__ void __launch_bounds__(T, 3 * 256 / T) k_sp_small(SpDev d, const int *__restrict__ list,
                                                             const double *__restrict__ Ax, double *__restrict__ F,
                                                             int *__restrict__ flag)
{
    extern __shared__ double S[];
    __shared__ double inv[DB];
    __shared__ short ki[KID_LDS][SPLU_SMALL];
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int ns = fr.ns, n = fr.nf, ld = n | 1;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    constexpr int NW = T / 64;
    /* the first entries' loads run beside the gather's */
    const bool e0 = tid < fr.nent;
    const uint32_t rc0 = e0 ? d.ent_rc[fr.ent + tid] : 0;
    const int src0 = e0 ? d.ent_src[fr.ent + tid] : 0;
    for (int q0 = 0; q0 == 0 || q0 < fr.nkid; q0 += KID_LDS) {
        const int nq = min(KID_LDS, fr.nkid - q0);
#pragma unroll
        for (int q = 0; q < KID_LDS; q++)
            if (tid < n) ki[q][tid] = q < nq ? (short)d.inv[fr.inv + (int64_t)(q0 + q) * n + tid] : (short)-1;
        /* an absent child is read as child 0 would be, and not taken */
        const double *base[KID_LDS];
        int kl[KID_LDS];
#pragma unroll
        for (int q = 0; q < KID_LDS; q++) {
            const SpluKid kd = nq > 0 ? d.kid[fr.kid0 + q0 + (q < nq ? q : 0)] : SpluKid{0, 0, 0, 0};
            base[q] = F + kd.schur;
            kl[q] = kd.ld;
        }
        __syncthreads();
        /* loads without a branch, so that a thread's are all in flight */
        auto gather = [&](auto kc) {
            constexpr int K = kc;
            for (int rb = 0; rb < n; rb += 64) {
                const int r = min(rb + lane, n - 1);
                int ir[K];
#pragma unroll
                for (int q = 0; q < K; q++) ir[q] = ki[q][r];
#pragma unroll 4
                for (int c = wv; c < n; c += NW) {
                    double t[K];
                    bool on[K];
#pragma unroll
                    for (int q = 0; q < K; q++) {
                        const int ic = ki[q][c];
                        on[q] = ic >= 0 && ir[q] >= 0;
                        t[q] = base[q][on[q] ? __mul24(ic, kl[q]) + ir[q] : 0];
                    }
                    double v = 0.0;
#pragma unroll
                    for (int q = 0; q < K; q++) v += on[q] ? t[q] : 0.0;
                    if (rb + lane < n) S[__mul24(c, ld) + r] = q0 ? S[__mul24(c, ld) + r] + v : v;
                }
            }
        };
        if (nq <= 0) {
            for (int e = tid; e < n * ld; e += T) S[e] = 0.0;
        } else if (nq <= 2) {
            gather(std::integral_constant<int, 2>());
        } else {
            gather(std::integral_constant<int, KID_LDS>());
        }
        __syncthreads();
    }
    if (e0) S[(rc0 >> 16) * ld + (rc0 & 0xffffu)] += Ax[src0];
    for (int e = tid + T; e < fr.nent; e += T) {
        const uint32_t rc = d.ent_rc[fr.ent + e];
        S[(rc >> 16) * ld + (rc & 0xffffu)] += Ax[d.ent_src[fr.ent + e]];
    }
    __syncthreads();
    double lmax = 0.0;
    bool bad = false;
    for (int kb = -DB; kb < ns; kb += DB) {   /* the first turn only factors block 0 */
        const int w = min(DB, ns - kb), t0 = kb + w;
        const bool more = t0 < ns;
        if (kb >= 0) {
            lmax = fmax(lmax, lds_solves(S, ld, kb, w, n, inv, wv, NW));
            __syncthreads();
        }
        /* wave 0 updates the next diagonal block and factors it while the
         * others update the rest */
        if (more && wv == 0) {
            if (kb >= 0) lds_tile<1>(S, ld, kb, w, n, &t0, &t0);
            bool b;
            lmax = fmax(lmax, diag_lu(S + t0 * ld + t0, ld, min(DB, ns - t0), inv, &b));
            bad |= b;
        } else if (kb >= 0) {
            lds_update(S, ld, kb, w, n, more ? wv - 1 : wv, more ? NW - 1 : NW, more);
        }
        __syncthreads();
    }
    double *Fr = F + fr.off;
    for (int c = wv; c < n; c += NW)
        for (int r = lane; r < n; r += 64) Fr[c * n + r] = S[c * ld + r];
    if (tid == 0 && bad) flag[0] = 1;
    report_lmax(lmax, flag);
}

/* columns SPLU_CG g .. of a larger front of few children: every entry the sum
 * over the children whose boundary holds its row and column (of those listed
 * as reaching these columns), then the CSC entries of these columns added */
__global__ void __launch_bounds__(WG) k_sp_asm(SpDev d, const int *__restrict__ list, const double *__restrict__ Ax,
                                               double *__restrict__ F)
{
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int g = blockIdx.y, n = fr.nf;
    const int cb = g * SPLU_CG, ce = min(cb + SPLU_CG, n);
    if (cb >= n || fr.up >= 0) return;
    double *Fr = F + fr.off;
    const int *inv = d.inv + fr.inv, *cg = d.cg + fr.cg + 2 * g, *gk = d.gk + fr.gk;
    for (int r = threadIdx.x; r < n; r += WG) {
        double v[SPLU_CG];
#pragma unroll
        for (int k = 0; k < SPLU_CG; k++) v[k] = 0.0;
        /* loads without a branch, so that a thread's 16 are all in flight */
        for (int s = cg[1]; s < cg[3]; s++) {
            const int q = gk[s];
            const int ir = inv[(int64_t)q * n + r];
            const SpluKid kd = d.kid[fr.kid0 + q];
            const double *Fc = F + kd.schur + max(ir, 0);
            double t[SPLU_CG];
            int ic[SPLU_CG];
#pragma unroll
            for (int k = 0; k < SPLU_CG; k++) {
                ic[k] = inv[(int64_t)q * n + min(cb + k, n - 1)];
                t[k] = Fc[(int64_t)max(ic[k], 0) * kd.ld];
            }
#pragma unroll
            for (int k = 0; k < SPLU_CG; k++) v[k] += ir >= 0 && ic[k] >= 0 ? t[k] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < SPLU_CG; k++)
            if (cb + k < ce) Fr[(int64_t)(cb + k) * n + r] = v[k];
    }
    __syncthreads();
    for (int e = cg[0] + (int)threadIdx.x; e < cg[2]; e += WG) {
        const uint32_t rc = d.ent_rc[fr.ent + e];
        Fr[(int64_t)(rc >> 16) * n + (rc & 0xffffu)] += Ax[d.ent_src[fr.ent + e]];
    }
}

/* a column of a larger front of many children, by one wavefront in LDS: the
 * children that hold the column add theirs, at their boundary's rows, one
 * after the other, KID_AHEAD of them loaded together; then the CSC entries.
 * The work is the children's entries, where by inverse lists it is every
 * child at every row: a system of 4732 fronts, most of them children of one of
 * 3089 unknowns, factors in 4.7 ms instead of 81 (32 with a launch a child). */
constexpr int KID_AHEAD = 4;
__global__ void __launch_bounds__(64) k_sp_asm_many(SpDev d, const int *__restrict__ list, const double *__restrict__ Ax,
                                                    double *__restrict__ F)
{
    extern __shared__ double acc[];
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int n = fr.nf, c = blockIdx.y, lane = threadIdx.x;
    if (c >= n) return;
    for (int r = lane; r < n; r += 64) acc[r] = 0.0;
    const SpluUp *up = d.up_ent + fr.upe;
    const int e0 = d.up_ptr[fr.up + c], e1 = d.up_ptr[fr.up + c + 1];
    for (int e = e0; e < e1; e += KID_AHEAD) {
        const double *col[KID_AHEAD];
        const int *rel[KID_AHEAD];
        int nb[KID_AHEAD], most = 0;
#pragma unroll
        for (int u = 0; u < KID_AHEAD; u++) {
            const SpluUp x = up[min(e + u, e1 - 1)];
            const SpluKid kd = d.kid[fr.kid0 + x.q];
            col[u] = F + kd.schur + (int64_t)x.i * kd.ld;
            rel[u] = d.rel + kd.wk;
            nb[u] = e + u < e1 ? kd.nb : 0;
            most = max(most, nb[u]);
        }
        for (int i0 = 0; i0 < most; i0 += 64) {
            const int i = i0 + lane;
            double v[KID_AHEAD];
            int r[KID_AHEAD];
#pragma unroll
            for (int u = 0; u < KID_AHEAD; u++) {
                const int j = min(i, max(nb[u] - 1, 0));
                v[u] = col[u][j];
                r[u] = rel[u][j];
            }
#pragma unroll
            for (int u = 0; u < KID_AHEAD; u++)
                if (i < nb[u]) acc[r[u]] += v[u];
        }
    }
    __syncthreads();
    const int *cg = d.cg + fr.cg + 2 * (c / SPLU_CG);
    for (int e = cg[0] + lane; e < cg[2]; e += 64) {
        const uint32_t rc = d.ent_rc[fr.ent + e];
        if ((int)(rc >> 16) == c) acc[rc & 0xffffu] += Ax[d.ent_src[fr.ent + e]];
    }
    __syncthreads();
    double *Fc = F + fr.off + (int64_t)c * n;
    for (int r = lane; r < n; r += 64) Fc[r] = acc[r];
}

/* Panel p of every front in list.  64 columns a launch, because a launch's time
 * is its chain of pivots and its latencies, and the next height's panels wait
 * for it: 42 us for 64 (the diagonal block ~20), where 32 took 41.  Every
 * workgroup factors the w x w
 * diagonal block for itself (a launch of its own would cost about as much as
 * this chain), by 16 pivots in LDS.  Then its wavefronts take the L21 rows
 * (X U11 = rows) and U12 columns (L11 X = columns) 64 at a time, one a lane
 * with its 64 entries in registers: the block's entries come 16 lanes a row
 * from LDS and are broadcast by DPP moves, with no barrier.  Workgroup 0 of a
 * front writes the block to dfac; the update launch copies it back, after
 * every workgroup of this launch has read the unfactored one. */
__global__ void __launch_bounds__(WG, 2) k_sp_panel(SpDev d, const int *__restrict__ list, int p,
                                                    double *__restrict__ F, double *__restrict__ dfac,
                                                    int *__restrict__ flag)
{
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int nsf = fr.ns, nf = fr.nf;
    const int kb = p * NB;
    if (kb >= nsf) return;
    const int w = min(NB, nsf - kb), t0 = kb + w, m = nf - t0, chunks = (m + 63) / 64;
    if (blockIdx.y > 0 && (int)blockIdx.y * (WG / 64) >= 2 * chunks) return;
    double *Fr = F + fr.off;
    __shared__ double D[NB * DLD];   /* [column][row] */
    __shared__ double inv[NB];
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    double lmax = 0.0;
    {
        double v[NB / (WG / 64)];   /* all in flight before the first is stored; zero beyond w */
#pragma unroll
        for (int q = 0; q < NB / (WG / 64); q++)
            v[q] = Fr[(int64_t)(kb + min(wv + q * (WG / 64), w - 1)) * nf + kb + min(lane, w - 1)];
#pragma unroll
        for (int q = 0; q < NB / (WG / 64); q++) {
            const int c = wv + q * (WG / 64);
            if (lane < NB) D[c * DLD + lane] = c < w && lane < w ? v[q] : 0.0;
        }
    }
    __syncthreads();
    const bool first = blockIdx.y == 0;
    auto factor = [&](int b) {
        bool bad;
        const double l = diag_lu(D + b * DLD + b, DLD, min(DB, w - b), inv + b, &bad);
        if (first) {
            lmax = fmax(lmax, l);
            if (bad && lane == 0) flag[0] = 1;
        }
    };
    for (int b = -DB; b < w; b += DB) {   /* the first turn only factors block 0 */
        const bool more = b + DB < w;
        if (!more) break;
        if (b >= 0) {
            const double l = lds_solves(D, DLD, b, DB, w, inv + b, wv, WG / 64);
            if (first) lmax = fmax(lmax, l);
            __syncthreads();
        }
        if (wv == 0) {
            const int nb = b + DB;
            if (b >= 0) lds_tile<1>(D, DLD, b, DB, w, &nb, &nb);
            factor(nb);
        } else if (b >= 0) {
            lds_update(D, DLD, b, DB, w, wv - 1, WG / 64 - 1, true);
        }
        __syncthreads();
    }
    if (first) {
        double *df = dfac + (int64_t)blockIdx.x * NB * NB;
        for (int c = wv; c < w; c += WG / 64)
            if (lane < w) df[c * w + lane] = D[c * DLD + lane];
    }
    const int it = (int)blockIdx.y * (WG / 64) + wv;
    if (it < 2 * chunks) {
        const bool row = it < chunks;
        const int t = (row ? it : it - chunks) * 64 + lane, i = t0 + min(t, m - 1), j = lane & (DB - 1);
        double *base = row ? Fr + (int64_t)kb * nf + i : Fr + (int64_t)i * nf + kb;
        const int64_t st = row ? nf : 1;
        double x[NB];
#pragma unroll
        for (int k = 0; k < NB; k++) x[k] = base[min(k, w - 1) * st];   /* beyond w: not used */
        asm volatile("" : "+v"(base));   /* the stores' addresses are formed again, not held */
        static_for<0, NB / DB>([&](auto bc) {
            constexpr int b = bc * DB;
            if (b < w) {
                /* what the pivots before take from these 16, then these 16 */
                const double iv = inv[b + j];
                auto operand = [&](int k) { return row ? D[(b + j) * DLD + k] : D[k * DLD + b + j]; };
                double un = operand(0);
                static_for<0, b + DB>([&](auto kc) {
                    constexpr int k = kc;
                    /* the next step's entries are read during this one, and
                     * no earlier: they would all be held at once */
                    const double u = un;
                    asm volatile("" ::: "memory");
                    if constexpr (k + 1 < b + DB) un = operand(k + 1);
                    if constexpr (k >= b) {
                        if (row) x[k] *= bcast16<k - b>(iv);
                    }
                    const double nx = -x[k];
                    static_for<(k >= b ? k - b + 1 : 0), DB>([&](auto qc) {
                        constexpr int q = qc;
                        x[b + q] = fma(bcast16<q>(u), nx, x[b + q]);
                        pin(x[b + q]);
                    });
                });
            }
        });
        if (t < m) {
            __attribute__((address_space(1))) double *p = (__attribute__((address_space(1))) double *)base;
#pragma unroll
            for (int k = 0; k < NB; k++)
                if (k < w) {
                    *p = x[k];
                    p += st;
                    if (row) lmax = fmax(lmax, fabs(x[k]));
                }
        }
    }
    report_lmax(lmax, flag);
}

/* F[t0:, t0:] -= L21 U12 for panel p, 64 x 64 tile blockIdx.y, 32 x 32 a
 * wave on the matrix cores, both operands staged 32 deep (38 KB: four
 * workgroups a CU cover each other's loads), with leading dimensions that
 * spread a wave's 4 depths and 16 rows or columns over the banks; block 0
 * also puts the factored diagonal block back from dfac. */
constexpr int TL = 64, KD = 32, LDL = 80, LDU = 36;
__global__ void __launch_bounds__(WG) k_sp_update(SpDev d, const int *__restrict__ list, int p,
                                                  double *__restrict__ F, const double *__restrict__ dfac)
{
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int nsf = fr.ns, nf = fr.nf;
    const int kb = p * NB;
    if (kb >= nsf) return;
    const int w = min(NB, nsf - kb), t0 = kb + w, m = nf - t0;
    double *Fr = F + fr.off;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    if (blockIdx.y == 0) {
        const double *df = dfac + (int64_t)blockIdx.x * NB * NB;
        for (int c = wv; c < w; c += WG / 64)
            if (lane < w) Fr[(int64_t)(kb + c) * nf + kb + lane] = df[c * w + lane];
    }
    const int T = (m + TL - 1) / TL;
    if ((int)blockIdx.y >= T * T) return;
    const int r0 = t0 + (blockIdx.y % T) * TL, c0 = t0 + (blockIdx.y / T) * TL;
    __shared__ double Ls[KD * LDL];   /* [depth][row] */
    __shared__ double Us[TL * LDU];   /* [column][depth] */
    const int li = lane & 15, lk = lane >> 4;
    const int rw = (wv & 1) * 32, cw = (wv >> 1) * 32;
    const bool live = r0 + rw < nf && c0 + cw < nf;
    d4 acc[2][2] = {};
    for (int k0 = 0; k0 < w; k0 += KD) {
        if (k0) __syncthreads();
#pragma unroll
        for (int q = 0; q < KD * 64 / WG; q++) {
            const int k = wv + q * (WG / 64), r = min(r0 + lane, nf - 1);
            const double v = Fr[(int64_t)(kb + min(k0 + k, w - 1)) * nf + r];
            Ls[k * LDL + lane] = k0 + k < w ? v : 0.0;
        }
#pragma unroll
        for (int q = 0; q < KD * 64 / WG; q++) {
            const int c = (tid >> 5) + q * (WG / 32), k = tid & 31;
            const double v = Fr[(int64_t)min(c0 + c, nf - 1) * nf + kb + min(k0 + k, w - 1)];
            Us[c * LDU + k] = k0 + k < w ? v : 0.0;
        }
        __syncthreads();
        if (live) {
#pragma unroll
            for (int q = 0; q < KD; q += 4) {
                const int k = q + lk;
                const double l0 = Ls[k * LDL + rw + li], l1 = Ls[k * LDL + rw + 16 + li];
                const double u0 = Us[(cw + li) * LDU + k], u1 = Us[(cw + 16 + li) * LDU + k];
                acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u0, l0, acc[0][0], 0, 0, 0);
                acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u0, l1, acc[0][1], 0, 0, 0);
                acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u1, l0, acc[1][0], 0, 0, 0);
                acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u1, l1, acc[1][1], 0, 0, 0);
            }
        }
    }
    if (!live) return;
    double cur[2][2][4];
#pragma unroll
    for (int cj = 0; cj < 2; cj++)
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int ri = 0; ri < 2; ri++)
                cur[cj][ri][v] = Fr[(int64_t)min(c0 + cw + 16 * cj + 4 * v + lk, nf - 1) * nf +
                                    min(r0 + rw + 16 * ri + li, nf - 1)];
#pragma unroll
    for (int cj = 0; cj < 2; cj++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int c = c0 + cw + 16 * cj + 4 * v + lk;
#pragma unroll
            for (int ri = 0; ri < 2; ri++) {
                const int r = r0 + rw + 16 * ri + li;
                if (r < nf && c < nf) Fr[(int64_t)c * nf + r] = cur[cj][ri][v] - acc[cj][ri][v];
            }
        }
}

__global__ void __launch_bounds__(WG) k_sp_perm(const int *__restrict__ rowsrc, const double *__restrict__ b,
                                                double *__restrict__ out, int n)
{
    const int r = blockIdx.x * WG + threadIdx.x;
    if (r < n) out[r] = b[rowsrc[r]];
}

/* Forward, a front's local unknown k before its own pivots: the right-hand
 * side where it is a pivot, and what the children's boundary parts (left in
 * the work vector wk, idx on, by their own forward step) hand up */
__device__ __forceinline__ double gather_rhs(const SpDev &d, const SpluFront &fr, int k, const double *bp,
                                             const double *wk)
{
    double v = k < fr.ns ? bp[d.idx[fr.idx + k]] : 0.0;
    if (fr.up >= 0) {
        const SpluUp *up = d.up_ent + fr.upe;
        const int e1 = d.up_ptr[fr.up + k + 1];
#pragma unroll 8
        for (int e = d.up_ptr[fr.up + k]; e < e1; e++) v += wk[d.kid[fr.kid0 + up[e].q].wk + up[e].i];
        return v;
    }
#pragma unroll 4
    for (int q = 0; q < fr.nkid; q++) {
        const int i = d.inv[fr.inv + (int64_t)q * fr.nf + k];
        if (i >= 0) v += wk[d.kid[fr.kid0 + q].wk + i];
    }
    return v;
}

constexpr int SR = (SPLU_SMALL + 63) / 64;   /* rows a lane holds of a small front */

/* count doubles to LDS, a workgroup's threads side by side, 16 loads each in
 * flight */
__device__ __forceinline__ void to_lds(double *S, const double *p, int count)
{
    for (int e0 = threadIdx.x; e0 < count; e0 += 16 * WG) {
        double v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = p[min(e0 + q * WG, count - 1)];
#pragma unroll
        for (int q = 0; q < 16; q++)
            if (e0 + q * WG < count) S[e0 + q * WG] = v[q];
    }
}

/* forward substitution of one small front a workgroup: its pivots' columns
 * are brought to LDS by all, then one wavefront holds the rows and takes a
 * column of L per step, with the pivot broadcast.  The chain is ~60 cycles a
 * pivot; loading its columns from memory 8 at a time as it went waited ~1 us
 * for every 8. */
__global__ void __launch_bounds__(WG) k_sp_fwd_small(SpDev d, const int *__restrict__ list,
                                                     const double *__restrict__ F, const double *__restrict__ bp,
                                                     double *__restrict__ wk, double *__restrict__ y)
{
    extern __shared__ double S[];   /* L's columns, ld nf; then the right-hand side */
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int ns = fr.ns, nf = fr.nf, lane = threadIdx.x & 63;
    double *r = S + ns * nf;
    if ((int)threadIdx.x < nf) r[threadIdx.x] = gather_rhs(d, fr, threadIdx.x, bp, wk);
    to_lds(S, F + fr.off, ns * nf);   /* the pivots' columns are contiguous */
    __syncthreads();
    if (wave_id() != 0) return;
    double v[SR];
    int row[SR];
#pragma unroll
    for (int q = 0; q < SR; q++) {
        row[q] = min(lane + 64 * q, nf - 1);
        v[q] = r[row[q]];
    }
#pragma unroll
    for (int s = 0; s < SR; s++) {
        const int ke = min(ns, 64 * s + 64);
        for (int k0 = 64 * s; k0 < ke; k0 += 8) {
            double l[8][SR];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int q = s; q < SR; q++)
                    if (64 * q < nf) l[j][q] = S[min(k0 + j, ns - 1) * nf + row[q]];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = k0 + j;
                if (k < ke) {
                    const double yk = rdlane(v[s], k & 63);
#pragma unroll
                    for (int q = s; q < SR; q++)
                        if (64 * q < nf && lane + 64 * q > k) v[q] -= l[j][q] * yk;
                }
            }
        }
    }
    const int *id = d.idx + fr.idx;
    double *w = wk + fr.idx;
#pragma unroll
    for (int q = 0; q < SR; q++) {
        const int k = lane + 64 * q;
        if (k < ns) y[id[k]] = v[q];
        else if (k < nf) w[k] = v[q];
    }
}

/* backward substitution of one small front a workgroup: the pivots' rows of
 * U to LDS (ld ns); y - U12 x of the boundary, its columns dealt to the four
 * wavefronts and their sums added in order; then the pivots from the last,
 * by one wavefront */
__global__ void __launch_bounds__(WG) k_sp_bwd_small(SpDev d, const int *__restrict__ list,
                                                     const double *__restrict__ F, const double *__restrict__ y,
                                                     double *__restrict__ x)
{
    extern __shared__ double S[];   /* U11; the boundary's x; the wavefronts' sums */
    constexpr int NW = WG / 64;
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int ns = fr.ns, nf = fr.nf, nb = nf - ns, lane = threadIdx.x & 63, wv = wave_id();
    const double *Fr = F + fr.off;
    const int *id = d.idx + fr.idx;
    double *xb = S + ns * ns, *part = xb + nb;
    int row[SR];
#pragma unroll
    for (int q = 0; q < SR; q++) row[q] = min(lane + 64 * q, ns - 1);
    if ((int)threadIdx.x < nb) xb[threadIdx.x] = x[id[ns + threadIdx.x]];
#pragma unroll
    for (int q = 0; q < SR; q++)   /* the columns of U11 a wavefront takes, 8 in flight */
        if (64 * q < ns)
            for (int c0 = wv; c0 < ns; c0 += 8 * NW) {
                double t[8];
#pragma unroll
                for (int j = 0; j < 8; j++) t[j] = Fr[(int64_t)min(c0 + j * NW, ns - 1) * nf + row[q]];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (c0 + j * NW < ns && lane + 64 * q < ns) S[(c0 + j * NW) * ns + lane + 64 * q] = t[j];
            }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SR; q++)
        if (64 * q < ns) {
            double a = 0.0;
            for (int c0 = wv; c0 < nb; c0 += 8 * NW) {
                double t[8];
#pragma unroll
                for (int j = 0; j < 8; j++) t[j] = Fr[(int64_t)(ns + min(c0 + j * NW, nb - 1)) * nf + row[q]];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (c0 + j * NW < nb) a += t[j] * xb[c0 + j * NW];
            }
            if (lane + 64 * q < ns) part[wv * ns + lane + 64 * q] = a;
        }
    __syncthreads();
    if (wv != 0) return;
    double v[SR], dg[SR], di[SR];
#pragma unroll
    for (int q = 0; q < SR; q++) {
        double a = part[row[q]];
#pragma unroll
        for (int w = 1; w < NW; w++) a += part[w * ns + row[q]];
        v[q] = y[id[row[q]]] - a;
        dg[q] = S[row[q] * ns + row[q]];
        di[q] = 1.0 / dg[q];
    }
    /* 64 pivots, from the last; EXACT divides, else quotients come from the
     * pivots' reciprocals.  num takes each lane's dividend. */
    auto pivots = [&](auto sc, auto exact, double &num) {
        constexpr int s = sc;
        const int ke = min(ns, 64 * s + 64);
        for (int k0 = ((ke - 1) & ~7); k0 >= 64 * s; k0 -= 8) {
            double u[8][SR];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int q = 0; q <= s; q++) u[j][q] = S[min(k0 + j, ns - 1) * ns + row[q]];
#pragma unroll
            for (int j = 7; j >= 0; j--) {
                const int k = k0 + j;
                if (k < ke) {
                    const double xk = rdlane(exact ? v[s] / dg[s] : div_by(v[s], dg[s], di[s]), k & 63);
#pragma unroll
                    for (int q = 0; q <= s; q++) {
                        const int i = lane + 64 * q;
                        if (i == k) {
                            num = v[q];
                            v[q] = xk;
                        } else if (i < k) {
                            v[q] -= u[j][q] * xk;
                        }
                    }
                }
            }
        }
    };
    static_for<0, SR>([&](auto rc) {
        constexpr int s = SR - 1 - rc;
        if (64 * s >= ns) return;
        double v0[s + 1], num = 1.0;
#pragma unroll
        for (int q = 0; q <= s; q++) v0[q] = v[q];
        pivots(std::integral_constant<int, s>(), std::false_type(), num);
        /* once more, dividing, where a quotient was out of div_by's range */
        if (__any(lane + 64 * s < ns && !div_by_ok(num, dg[s]))) {
#pragma unroll
            for (int q = 0; q <= s; q++) v[q] = v0[q];
            pivots(std::integral_constant<int, s>(), std::true_type(), num);
        }
    });
#pragma unroll
    for (int q = 0; q < SR; q++)
        if (lane + 64 * q < ns) x[id[lane + 64 * q]] = v[q];
}

/* Panel p forward: the 64 pivots solved by wave 0 of every workgroup (one
 * row a lane, the solved pivot broadcast), then each of the workgroup's 256
 * rows below takes its 64 products.  Its loads need nothing of the triangle
 * and are issued before it.  Panel 0 gathers the rows (a launch of its own
 * for that cost 6 us a height), the others find them in wk. */
__global__ void __launch_bounds__(WG) k_sp_fwd_blk(SpDev d, const int *__restrict__ list, int p,
                                                   const double *__restrict__ F, const double *__restrict__ bp,
                                                   double *wk, double *__restrict__ y)
{
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int nsf = fr.ns, nf = fr.nf;
    const int kb = p * NB;
    if (kb >= nsf) return;
    const int w = min(NB, nsf - kb), t0 = kb + w;
    if (blockIdx.y > 0 && t0 + (int)blockIdx.y * WG >= nf) return;
    __shared__ double yb[NB];
    const double *Fr = F + fr.off;
    double *wf = wk + fr.idx;
    const int tid = threadIdx.x;
    const int i = t0 + blockIdx.y * WG + tid, ic = min(i, nf - 1);
    double l[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) l[k] = k < w ? Fr[(int64_t)(kb + k) * nf + ic] : 0.0;
    double ri = p == 0 ? gather_rhs(d, fr, ic, bp, wk) : wf[ic];
    if (tid < 64) {
        double lv[NB];
        const int row = kb + min(tid, w - 1);
#pragma unroll
        for (int k = 0; k < NB; k++) lv[k] = k < w ? Fr[(int64_t)(kb + k) * nf + row] : 0.0;
        double v = p == 0 ? gather_rhs(d, fr, row, bp, wk) : wf[row];
        if (tid >= w) v = 0.0;
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const double yk = rdlane(v, k);
            if (tid > k) v -= lv[k] * yk;
        }
        yb[tid] = tid < w ? v : 0.0;
        if (blockIdx.y == 0 && tid < w) y[d.idx[fr.idx + kb + tid]] = v;
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NB; k++) s += l[k] * yb[k];
    ri -= s;
    if (i < nf) wf[i] = ri;
}

constexpr int OFF_ROWS = 64;    /* rows per workgroup of the boundary products */
constexpr int OFF_WG = 1024;

/* wk_f = y_f - U12 x_boundary for the larger fronts of one height (ancestors
 * solved): 64 pivot rows per workgroup, its 16 waves on interleaved 64-column
 * slices; the partial sums are added in wave order, so the result does not
 * depend on timing */
__global__ void __launch_bounds__(OFF_WG) k_sp_bwd_off(SpDev d, const int *__restrict__ list,
                                                       const double *__restrict__ F, const double *__restrict__ y,
                                                       const double *__restrict__ x, double *__restrict__ wk)
{
    __shared__ double xv[OFF_WG];
    __shared__ double part[OFF_WG / 64][OFF_ROWS];
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int nsf = fr.ns, nf = fr.nf, nbf = nf - nsf;
    if ((int)blockIdx.y * OFF_ROWS >= nsf) return;
    const double *Fr = F + fr.off;
    const int *id = d.idx + fr.idx;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    const int i = blockIdx.y * OFF_ROWS + lane;
    const int ir = min(i, nsf - 1);
    double s = 0.0;
    for (int j0 = 0; j0 < nbf; j0 += OFF_WG) {
        __syncthreads();
        xv[tid] = j0 + tid < nbf ? x[id[nsf + j0 + tid]] : 0.0;
        __syncthreads();
        const int js = j0 + wv * 64;
        const int jn = min(64, nbf - js);
        const double *col = Fr + (int64_t)(nsf + js) * nf + ir;
#pragma unroll 16
        for (int j = 0; j < jn; j++) s += col[(int64_t)j * nf] * xv[wv * 64 + j];
    }
    part[wv][lane] = s;
    __syncthreads();
    if (wv == 0 && i < nsf) {
        double t = part[0][lane];
#pragma unroll
        for (int q = 1; q < OFF_WG / 64; q++) t += part[q][lane];
        wk[fr.idx + i] = y[id[i]] - t;
    }
}

/* panel p backward, as k_sp_fwd_blk: the 64 pivots from the last, then 256
 * rows above per workgroup.  A front without a boundary starts from y, the
 * others from what k_sp_bwd_off left in wk. */
__global__ void __launch_bounds__(WG) k_sp_bwd_blk(SpDev d, const int *__restrict__ list, int p,
                                                   const double *__restrict__ F, const double *__restrict__ y,
                                                   double *__restrict__ wk, double *__restrict__ x)
{
    const SpluFront fr = d.front[list[blockIdx.x]];
    const int nsf = fr.ns, nf = fr.nf;
    const int kb = p * NB;
    if (kb >= nsf) return;
    const int w = min(NB, nsf - kb);
    if (blockIdx.y > 0 && (int)blockIdx.y * WG >= kb) return;
    __shared__ double xb[NB];
    const double *Fr = F + fr.off;
    double *wf = wk + fr.idx;
    const int tid = threadIdx.x;
    const int i = blockIdx.y * WG + tid, ic = min(i, max(kb - 1, 0));
    double u[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) u[k] = k < w ? Fr[(int64_t)(kb + k) * nf + ic] : 0.0;
    const bool fresh = nf == nsf && kb + NB >= nsf;
    const int *id = d.idx + fr.idx;
    double ri = fresh ? y[id[ic]] : wf[ic];
    if (tid < 64) {
        double uv[NB];
        const int row = min(tid, w - 1);
#pragma unroll
        for (int k = 0; k < NB; k++) uv[k] = k < w ? Fr[(int64_t)(kb + k) * nf + kb + row] : 0.0;
        const double dg = Fr[(int64_t)(kb + row) * nf + kb + row], di = 1.0 / dg;
        const double v0 = tid < w ? (fresh ? y[id[kb + row]] : wf[kb + row]) : 0.0;
        double v = v0, num = 1.0;
        auto pivots = [&](auto exact) {
#pragma unroll
            for (int k = NB - 1; k >= 0; k--) {
                if (k < w) {
                    const double xk = rdlane(exact ? v / dg : div_by(v, dg, di), k);
                    if (tid == k) {
                        num = v;
                        v = xk;
                    } else if (tid < k) {
                        v -= uv[k] * xk;
                    }
                }
            }
        };
        pivots(std::false_type());
        if (__any(tid < w && !div_by_ok(num, dg))) {   /* as k_sp_bwd_small */
            v = v0;
            pivots(std::true_type());
        }
        xb[tid] = tid < w ? v : 0.0;
        if (blockIdx.y == 0 && tid < w) x[id[kb + tid]] = v;
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NB; k++) s += u[k] * xb[k];
    ri -= s;
    if (i < kb) wf[i] = ri;
}

enum { L_SMALL, L_ASM, L_ASM_MANY, L_PANEL, L_UPDATE, L_FWD_SMALL, L_FWD_DBK, L_BWD_SMALL, L_BWD_OFF, L_BWD_DBK };
/* a launch: fronts lev[first ..+gx) (L_ASM_MANY: of the list of those with many
 * children), panel p, gy workgroups a front, dynamic LDS */
struct Step {
    int kind, first, p;
    unsigned gx, gy;
    size_t lds;
};

template <class T>
int upload(T **dst, const std::vector<T> &v)
{
    const size_t bytes = std::max<size_t>(1, v.size()) * sizeof(T);
    NGMI_HIP(hipMalloc((void **)dst, bytes));
    if (!v.empty()) NGMI_HIP(hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return NGMI_OK;
}

}  // namespace

struct ngmi_splu {
    SpluSym S;
    bool ready = false;      /* device buffers allocated and plan built */
    bool factored = false;   /* the last ngmi_splu_factor succeeded */
    double lmax = 0.0;       /* its largest |l| multiplier */
    SpDev d{};
    std::vector<void *> bufs;
    int *d_lev = nullptr, *d_many = nullptr, *d_rowsrc = nullptr, *d_flag = nullptr;
    double *F = nullptr, *dfac = nullptr, *wk = nullptr, *vb = nullptr, *vy = nullptr, *vx = nullptr;
    std::vector<Step> factor, fwd, bwd;
};

/* frees every device buffer, so a later splu_device call starts from nothing */
static void splu_release(ngmi_splu *s)
{
    for (void *p : s->bufs) (void)hipFree(p);
    s->bufs.clear();
    s->factor.clear();
    s->fwd.clear();
    s->bwd.clear();
    s->ready = false;
    s->factored = false;
}

static int splu_device_alloc(ngmi_splu *s);

static int splu_device(ngmi_splu *s)
{
    if (s->ready) return NGMI_OK;
    const int rc = splu_device_alloc(s);
    if (rc != NGMI_OK) splu_release(s);
    return rc;
}

static int splu_device_alloc(ngmi_splu *s)
{
    const SpluSym &S = s->S;
    int rc;
    auto put = [&](auto &dst, const auto &v) {
        std::remove_const_t<std::remove_pointer_t<std::remove_reference_t<decltype(dst)>>> *p = nullptr;
        const int r = upload(&p, v);
        if (p) s->bufs.push_back(p);
        dst = p;
        return r;
    };
    auto room = [&](auto &dst, size_t count) -> int {
        void *p = nullptr;
        NGMI_HIP(hipMalloc(&p, std::max<size_t>(1, count) * sizeof(*dst)));
        s->bufs.push_back(p);
        dst = static_cast<std::remove_reference_t<decltype(dst)>>(p);
        return NGMI_OK;
    };
#define DO(call) \
    if ((rc = (call)) != NGMI_OK) return rc
    DO(put(s->d.front, S.front));
    DO(put(s->d.kid, S.kid));
    DO(put(s->d.idx, S.idx));
    DO(put(s->d.ent_src, S.ent_src));
    DO(put(s->d.ent_rc, S.ent_rc));
    DO(put(s->d.cg, S.cg));
    DO(put(s->d.gk, S.gk));
    DO(put(s->d.inv, S.inv));
    DO(put(s->d.up_ptr, S.up_ptr));
    DO(put(s->d.up_ent, S.up_ent));
    DO(put(s->d.rel, S.up_ptr.empty() ? std::vector<int>() : S.rel));
    DO(put(s->d_lev, S.lev));
    DO(put(s->d_rowsrc, S.rowsrc));
    DO(room(s->d_flag, 4));   /* zero-pivot flag, pad, largest |l| */
    DO(room(s->F, (size_t)S.store));
    DO(room(s->wk, S.idx.size()));
    DO(room(s->vb, (size_t)S.n));
    DO(room(s->vy, (size_t)S.n));
    DO(room(s->vx, (size_t)S.n));

    /* launch plan by height */
    auto size = [&](int q) { return S.ns[S.lev[q]] + S.nb[S.lev[q]]; };
    auto small_lds = [](int n) { return (size_t)n * (n | 1) * sizeof(double); };
    std::vector<Step> back;   /* the backward solve's launches, leaves first */
    std::vector<int> many;    /* larger fronts of many children, by height */
    int most = 1;
    for (int h = 0; h <= S.H; h++) {
        const int b = S.lev_ptr[h], e = S.lev_ptr[h + 1];
        int big = b;
        while (big < e && size(big) <= SPLU_SMALL) big++;
        /* small fronts: a launch for each size that lets another workgroup
         * share a CU's LDS (4 up to 70 unknowns, 3 up to 80, 2 up to 99),
         * but one for all when there is no more than a front to each of the
         * 256 CUs, where sharing gains nothing */
        for (int q = b; q < big;) {
            int r = big;
            if (big - b > 256)
                for (int limit : {70, 80, 99})
                    if (size(q) <= limit) {
                        r = q;
                        while (r < big && size(r) <= limit) r++;
                        break;
                    }
            /* eight waves where the LDS leaves room for one or two fronts */
            s->factor.push_back({L_SMALL, q, size(r - 1) > 80, (unsigned)(r - q), 1, small_lds(size(r - 1))});
            size_t lf = 0, lb = 0;
            for (int i = q; i < r; i++) {
                const size_t ns = S.ns[S.lev[i]], nf = size(i);
                lf = std::max(lf, (ns * nf + nf) * sizeof(double));
                lb = std::max(lb, (ns * ns + nf - ns + WG / 64 * ns) * sizeof(double));
            }
            s->fwd.push_back({L_FWD_SMALL, q, 0, (unsigned)(r - q), 1, lf});
            back.push_back({L_BWD_SMALL, q, 0, (unsigned)(r - q), 1, lb});
            q = r;
        }
        if (big == e) continue;
        const unsigned nl = (unsigned)(e - big);
        most = std::max(most, e - big);
        int maxns = 0, maxnb = 0, manynf = 0;
        const int many0 = (int)many.size();
        for (int q = big; q < e; q++) {
            maxns = std::max(maxns, S.ns[S.lev[q]]);
            maxnb = std::max(maxnb, S.nb[S.lev[q]]);
            if (S.front[S.lev[q]].up < 0) continue;
            many.push_back(S.lev[q]);
            manynf = std::max(manynf, size(q));
        }
        const int maxnf = size(e - 1);
        s->factor.push_back({L_ASM, big, 0, nl, (unsigned)((maxnf + SPLU_CG - 1) / SPLU_CG), 0});
        if (manynf)
            s->factor.push_back({L_ASM_MANY, many0, 0, (unsigned)many.size() - many0, (unsigned)manynf,
                                 manynf * sizeof(double)});
        std::vector<Step> bb;
        for (int p = 0; p * NB < maxns; p++) {
            int64_t chunks = 1, tiles = 1, below = 1;
            for (int q = big; q < e; q++) {
                const int f = S.lev[q];
                if (p * NB >= S.ns[f]) continue;
                const int64_t m = size(q) - (p * NB + std::min(NB, S.ns[f] - p * NB));
                const int64_t T = (m + TL - 1) / TL;
                chunks = std::max(chunks, (2 * ((m + 63) / 64) + WG / 64 - 1) / (WG / 64));
                below = std::max(below, (m + WG - 1) / WG);
                tiles = std::max(tiles, T * T);
            }
            if (tiles > 65535) {
                set_error("splu: front too large for the launch grid");
                return NGMI_E_UNSUPP;
            }
            s->factor.push_back({L_PANEL, big, p, nl, (unsigned)chunks, 0});
            s->factor.push_back({L_UPDATE, big, p, nl, (unsigned)tiles, 0});
            s->fwd.push_back({L_FWD_DBK, big, p, nl, (unsigned)below, 0});
            bb.push_back({L_BWD_DBK, big, p, nl, (unsigned)std::max(1, (p * NB + WG - 1) / WG), 0});
        }
        back.insert(back.end(), bb.begin(), bb.end());
        if (maxnb) back.push_back({L_BWD_OFF, big, 0, nl, (unsigned)((maxns + OFF_ROWS - 1) / OFF_ROWS), 0});
    }
    s->bwd.assign(back.rbegin(), back.rend());
    DO(put(s->d_many, many));
    DO(room(s->dfac, (size_t)most * NB * NB));
#undef DO
    NGMI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sp_small<256>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)small_lds(SPLU_SMALL)));
    NGMI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sp_small<512>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)small_lds(SPLU_SMALL)));
    constexpr size_t n = SPLU_SMALL;   /* the most a small front's solves take, at ns = nf = n */
    NGMI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sp_fwd_small),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)((n * n + n) * sizeof(double))));
    NGMI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sp_bwd_small),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)((n * n + WG / 64 * n) * sizeof(double))));
    s->ready = true;
    return NGMI_OK;
}

extern "C" {

int ngmi_splu_analyze(int n, const int64_t *Ap, const int *Ai, ngmi_splu **out)
{
    if (!out) return NGMI_E_PANIC;
    *out = nullptr;
    ngmi_splu *s = new ngmi_splu();
    const int rc = splu_analyze(n, Ap, Ai, s->S);
    if (rc != NGMI_OK) {
        delete s;
        return rc;
    }
    *out = s;
    return NGMI_OK;
}

void ngmi_splu_free(ngmi_splu *s)
{
    if (!s) return;
    splu_release(s);
    delete s;
}

int ngmi_splu_info(const ngmi_splu *s, int64_t *fronts, int64_t *heights, int64_t *max_front,
                   int64_t *front_doubles, int64_t *lu_nonzeros, double *flops)
{
    if (!s) return NGMI_E_PANIC;
    if (fronts) *fronts = s->S.nf;
    if (heights) *heights = s->S.H + 1;
    if (max_front) *max_front = s->S.max_front;
    if (front_doubles) *front_doubles = s->S.store;
    if (lu_nonzeros) *lu_nonzeros = s->S.lu_nnz;
    if (flops) *flops = s->S.flops;
    return NGMI_OK;
}

int ngmi_splu_front(const ngmi_splu *s, int f, int *ns, int *nb, int *parent, int *idx)
{
    if (!s || f < 0 || f >= s->S.nf) {
        set_error("splu_front: no front %d", f);
        return NGMI_E_PARMVAL;
    }
    const SpluSym &S = s->S;
    if (ns) *ns = S.ns[f];
    if (nb) *nb = S.nb[f];
    if (parent) *parent = S.parent[f];
    if (idx) std::copy(S.idx.begin() + S.idx_off[f], S.idx.begin() + S.idx_off[f + 1], idx);
    return NGMI_OK;
}

int ngmi_splu_rowsrc(const ngmi_splu *s, int *rowsrc)
{
    if (!s || !rowsrc) return NGMI_E_PANIC;
    std::copy(s->S.rowsrc.begin(), s->S.rowsrc.end(), rowsrc);
    return NGMI_OK;
}

int ngmi_splu_factor(ngmi_splu *s, const double *Ax, void *stream)
{
    if (!s || !Ax) return NGMI_E_PANIC;
    int rc = splu_device(s);
    if (rc != NGMI_OK) return rc;
    s->factored = false;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_sp_clear, dim3(1), dim3(64), 0, st, s->d_flag);
    for (const Step &p : s->factor) {
        const int *list = s->d_lev + p.first;   /* not L_ASM_MANY's */
        const dim3 g(p.gx, p.gy), wg(WG);
        if (p.kind == L_SMALL && p.p)
            hipLaunchKernelGGL(k_sp_small<512>, g, dim3(512), p.lds, st, s->d, list, Ax, s->F, s->d_flag);
        else if (p.kind == L_SMALL)
            hipLaunchKernelGGL(k_sp_small<256>, g, wg, p.lds, st, s->d, list, Ax, s->F, s->d_flag);
        else if (p.kind == L_ASM) hipLaunchKernelGGL(k_sp_asm, g, wg, 0, st, s->d, list, Ax, s->F);
        else if (p.kind == L_ASM_MANY)
            hipLaunchKernelGGL(k_sp_asm_many, g, dim3(64), p.lds, st, s->d, s->d_many + p.first, Ax, s->F);
        else if (p.kind == L_PANEL)
            hipLaunchKernelGGL(k_sp_panel, g, wg, 0, st, s->d, list, p.p, s->F, s->dfac, s->d_flag);
        else hipLaunchKernelGGL(k_sp_update, g, wg, 0, st, s->d, list, p.p, s->F, s->dfac);
    }
    NGMI_HIP(hipGetLastError());
    int fl[4] = {0, 0, 0, 0};
    NGMI_HIP(hipMemcpyAsync(fl, s->d_flag, sizeof(fl), hipMemcpyDeviceToHost, st));
    NGMI_HIP(hipStreamSynchronize(st));
    std::memcpy(&s->lmax, fl + 2, sizeof(double));
    if (fl[0]) {
        set_error("splu_factor: zero or non-finite pivot");
        return NGMI_E_SINGULAR;
    }
    s->factored = true;
    return NGMI_OK;
}

int ngmi_splu_multiplier(const ngmi_splu *s, double *lmax)
{
    if (!s || !lmax) return NGMI_E_PANIC;
    if (!s->factored) {
        set_error("splu_multiplier: no successful factorization");
        return NGMI_E_SINGULAR;
    }
    *lmax = s->lmax;
    return NGMI_OK;
}

int ngmi_splu_solve(ngmi_splu *s, double *b, void *stream)
{
    if (!s || !b) return NGMI_E_PANIC;
    if (!s->ready || !s->factored) {
        set_error("splu_solve: no successful factorization");
        return NGMI_E_SINGULAR;
    }
    const SpluSym &S = s->S;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_sp_perm, dim3((S.n + WG - 1) / WG), dim3(WG), 0, st, s->d_rowsrc, b, s->vb, S.n);
    for (const Step &p : s->fwd) {
        const int *list = s->d_lev + p.first;
        const dim3 g(p.gx, p.gy);
        if (p.kind == L_FWD_SMALL)
            hipLaunchKernelGGL(k_sp_fwd_small, g, dim3(WG), p.lds, st, s->d, list, s->F, s->vb, s->wk, s->vy);
        else hipLaunchKernelGGL(k_sp_fwd_blk, g, dim3(WG), 0, st, s->d, list, p.p, s->F, s->vb, s->wk, s->vy);
    }
    for (const Step &p : s->bwd) {
        const int *list = s->d_lev + p.first;
        const dim3 g(p.gx, p.gy);
        if (p.kind == L_BWD_SMALL)
            hipLaunchKernelGGL(k_sp_bwd_small, g, dim3(WG), p.lds, st, s->d, list, s->F, s->vy, s->vx);
        else if (p.kind == L_BWD_OFF)
            hipLaunchKernelGGL(k_sp_bwd_off, g, dim3(OFF_WG), 0, st, s->d, list, s->F, s->vy, s->vx, s->wk);
        else hipLaunchKernelGGL(k_sp_bwd_blk, g, dim3(WG), 0, st, s->d, list, p.p, s->F, s->vy, s->wk, s->vx);
    }
    NGMI_HIP(hipGetLastError());
    NGMI_HIP(hipMemcpyAsync(b, s->vx, (size_t)S.n * sizeof(double), hipMemcpyDeviceToDevice, st));
    return NGMI_OK;
}

}  // extern "C"
