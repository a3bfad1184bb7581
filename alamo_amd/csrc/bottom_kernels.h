// bottom_kernels.h -- single-workgroup bottom solvers for the coarsest MG level.
//
// The coarsest level of the hierarchy holds 3^3 nodes for power-of-two
// boxes, so the whole bottom solve (BiCGStab with the operator diagonal as
// left preconditioner, then the post-smoothing of a failed solve) runs in one
// workgroup: no host round trips and no launch per BiCGStab step.
// Restates amrex::MLMG::actualBottomSolve + MLCGSolver::solve_bicgstab with
// Operator<Grid::Node>::normalize (src/Operator/Operator.cpp:156-165) and the
// bicgstab choice of src/Solver/Nonlocal/Linear.H:258.
#pragma once
#include "elastic_kernels.h"

namespace ael {

constexpr int kBottomBlock = 1024;

// Block-wide max (op 0) or sum (op 1); every thread returns the same value.
__device__ __forceinline__ double block_reduce(double v, int op, double* red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off);
        v = op == 0 ? fmax(v, o) : v + o;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double r = 0.0;
    for (int q = 0; q < nw; ++q) r = op == 0 ? fmax(r, red[q]) : r + red[q];
    return r;
}

template <int SYM>
__device__ void blk_apply(const double* __restrict__ in, double* __restrict__ out, const double* __restrict__ C,
                          const int* __restrict__ bct, int uniform, const Lvl& L) {
    for (long id = threadIdx.x; id < L.N; id += blockDim.x) {
        int i, j, k;
        node_ijk(id, L, i, j, k);
        double o[3];
        apply_node<double, SYM>(in, C, bct, uniform, L, i, j, k, id, o);
        out[id] = o[0];
        out[L.N + id] = o[1];
        out[2 * L.N + id] = o[2];
    }
    __syncthreads();
}

// w: 10 vectors of 3N doubles of scratch.  status[0] receives the BiCGStab
// return code (0 converged, 1..4 breakdown, 8 not converged).
template <int SYM>
__global__ void __launch_bounds__(kBottomBlock)
    k_bottom_solve(double* __restrict__ x, const double* __restrict__ rhs, const double* __restrict__ C,
                   const double* __restrict__ diag, const int* __restrict__ bct, int uniform, Lvl L, double omega,
                   int maxiter, double eps_rel, int nuf, double* __restrict__ w, int* __restrict__ status) {
    __shared__ double red[kBottomBlock / 64];
    const long M = 3 * L.N;
    double *ph = w, *sh = w + M, *p = w + 2 * M, *r = w + 3 * M, *s = w + 4 * M, *rh = w + 5 * M, *v = w + 6 * M,
           *t = w + 7 * M, *tmp = w + 8 * M;
    const int tid = threadIdx.x, nt = blockDim.x;
    // actualBottomSolve: x = 0; MLCGSolver: r = b - A x, normalized.
    for (long q = tid; q < M; q += nt) x[q] = 0.0;
    __syncthreads();
    blk_apply<SYM>(x, v, C, bct, uniform, L);
    double loc = 0.0;
    for (long q = tid; q < M; q += nt) {
        const double rq = (rhs[q] + (-1.0) * v[q]) / diag[q];
        r[q] = rq;
        rh[q] = rq;
        loc = fmax(loc, fabs(rq));
    }
    const double rnorm0 = block_reduce(loc, 0, red);
    double rnorm = rnorm0, rho_1 = 0.0, alpha = 0.0, omg = 0.0;
    int ret = 0;
    if (rnorm0 != 0.0) {
        for (int iter = 1; iter <= maxiter; ++iter) {
            loc = 0.0;
            for (long q = tid; q < M; q += nt) loc += rh[q] * r[q];
            const double rho = block_reduce(loc, 1, red);
            if (rho == 0.0) { ret = 1; break; }
            if (iter == 1) {
                for (long q = tid; q < M; q += nt) p[q] = r[q];
            } else {
                const double beta = (rho / rho_1) * (alpha / omg);
                for (long q = tid; q < M; q += nt) {
                    const double pq = p[q] + (-omg) * v[q];
                    p[q] = r[q] + beta * pq;
                }
            }
            for (long q = tid; q < M; q += nt) ph[q] = p[q];
            __syncthreads();
            blk_apply<SYM>(ph, v, C, bct, uniform, L);
            loc = 0.0;
            for (long q = tid; q < M; q += nt) {
                v[q] /= diag[q];
                loc += rh[q] * v[q];
            }
            const double rhTv = block_reduce(loc, 1, red);
            if (rhTv != 0.0) alpha = rho / rhTv;
            else { ret = 2; break; }
            loc = 0.0;
            for (long q = tid; q < M; q += nt) {
                x[q] += alpha * ph[q];
                const double sq = 1.0 * r[q] + (-alpha) * v[q];
                s[q] = sq;
                sh[q] = sq;
                loc = fmax(loc, fabs(sq));
            }
            rnorm = block_reduce(loc, 0, red);
            if (rnorm < eps_rel * rnorm0) break;
            blk_apply<SYM>(sh, t, C, bct, uniform, L);
            double l1 = 0.0, l2 = 0.0;
            for (long q = tid; q < M; q += nt) {
                t[q] /= diag[q];
                l1 += t[q] * t[q];
                l2 += t[q] * s[q];
            }
            const double tt = block_reduce(l1, 1, red);
            const double ts = block_reduce(l2, 1, red);
            if (tt != 0.0) omg = ts / tt;
            else { ret = 3; break; }
            loc = 0.0;
            for (long q = tid; q < M; q += nt) {
                x[q] += omg * sh[q];
                const double rq = 1.0 * s[q] + (-omg) * t[q];
                r[q] = rq;
                loc = fmax(loc, fabs(rq));
            }
            rnorm = block_reduce(loc, 0, red);
            if (rnorm < eps_rel * rnorm0) break;
            if (omg == 0.0) { ret = 4; break; }
            rho_1 = rho;
        }
        if (ret == 0 && rnorm > eps_rel * rnorm0) ret = 8;
        // sorig is the zero initial guess: keep x only when it reduced the residual
        if (!((ret == 0 || ret == 8) && rnorm < rnorm0))
            for (long q = tid; q < M; q += nt) x[q] = 0.0;
        // actualBottomSolve: a failed solve (ret other than 0, 9) is discarded
        if (ret != 0 && ret != 9)
            for (long q = tid; q < M; q += nt) x[q] = 0.0;
        __syncthreads();
        // then nuf Fsmooth calls after a failure (nub = 0 after success)
        const int nsm = ret == 0 ? 0 : nuf;
        for (int sm = 0; sm < 2 * nsm; ++sm) {
            const double* xin = (sm & 1) ? tmp : x;
            double* xout = (sm & 1) ? x : tmp;
            blk_apply<SYM>(xin, v, C, bct, uniform, L);
            for (long q = tid; q < M; q += nt) {
                const double xv = xin[q], dv = diag[q];
                const double Rx = v[q] - xv * dv;
                xout[q] = (1.0 - omega) * xv + omega * (rhs[q] - Rx) / dv;
            }
            __syncthreads();
        }
    }
    if (tid == 0) status[0] = ret;
}

// --- The bottom solve on the assembled rows of the coarsest operator ------
// The rows of a coarsest level with at most kDenseMax unknowns, without their
// zeros.  A row of the operator touches the 19 nodes of its stencil (a
// boundary row at most 7, a wrapped row the same 19), so the three rows of a
// node share at most 57 columns.  Slot u of the kRowSlots of a node holds a
// column (its component and node, cols) and the three rows' values there over
// the rows' diagonal (vals); kRowHalf slots go to each of the two threads that
// work on the node, which read vals[((r * kRowHalf + k) * N + node) * 2 + half].
constexpr int kRowSlots = 58, kRowHalf = kRowSlots / 2;

// One wave per node: its columns in ascending order from the dense operator A
// (column-major, M x M), 64 candidates at a time.  A node with more than
// kRowSlots columns would break the bound above: its values become NaN, which
// the solve reports.
__global__ void __launch_bounds__(64) k_bottom_rows(const double* __restrict__ A, const double* __restrict__ diag, int N,
                                                    double* __restrict__ vals, unsigned short* __restrict__ cols) {
    const int node = (int)blockIdx.x, M = 3 * N, lane = (int)threadIdx.x;
    const double d[3] = {diag[node], diag[N + node], diag[2 * N + node]};
    auto put = [&](int u, int c, const double a[3]) {
        const int half = u / kRowHalf, k = u - half * kRowHalf;
        const long at = ((long)k * N + node) * 2 + half, plane = 2L * kRowHalf * N;
        cols[at] = (unsigned short)c;
        for (int r = 0; r < 3; ++r) vals[at + r * plane] = a[r];
    };
    int n = 0;
    for (int c0 = 0; c0 < M; c0 += 64) {
        const int c = c0 + lane;
        double a[3];
        for (int r = 0; r < 3; ++r) a[r] = c < M ? A[(long)c * M + r * N + node] : 0.0;
        const bool have = a[0] != 0.0 || a[1] != 0.0 || a[2] != 0.0;
        const unsigned long long bal = __ballot(have);
        const int u = n + (int)__popcll(bal & (lane ? ~0ull >> (64 - lane) : 0ull));
        if (have && u < kRowSlots) {
            for (int r = 0; r < 3; ++r) a[r] /= d[r];
            put(u, c, a);
        }
        n += (int)__popcll(bal);
    }
    const bool over = n > kRowSlots;
    const double pad[3] = {over ? __longlong_as_double(0x7ff8000000000000ll) : 0.0, 0.0, 0.0};
    for (int u = (over ? 0 : n) + lane; u < kRowSlots; u += 64) put(u, node, pad);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// Sum (MAX false) or max over a full wave, the same value in every lane: within
// rows of 16 lanes by DPP, the four rows through scalar registers (no LDS).
template <bool MAX>
__device__ __forceinline__ double wave_all(double v) {
    auto op = [](double a, double b) { return MAX ? fmax(a, b) : a + b; };
    v = op(v, dpp_f64<0xB1>(v));   // lane ^ 1
    v = op(v, dpp_f64<0x4E>(v));   // lane ^ 2
    v = op(v, dpp_f64<0x141>(v));  // the other four of eight
    v = op(v, dpp_f64<0x140>(v));  // the other eight of sixteen
    return op(op(readlane_f64(v, 0), readlane_f64(v, 16)), op(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// BiCGStab with the diagonal as left preconditioner, then the smoothing of a
// failed solve (the algorithm of k_bottom_solve), by one workgroup.  The solve
// is a chain of products and dot products, so its time is the latency of one
// step, not bytes: two threads a node hold that node's rows in registers
// (kBottomRegN nodes and fewer; above, they stream from L2), its three rows
// share the gathers, and the norm and the dots that a step forms at one point
// share a reduction (5 barriers a step).  Measured at 360 unknowns (the bottom of a box of
// 65 x 49 x 81 nodes): 122 us a solve, where products with the dense operator
// (one row a thread, its columns from L2, a reduction for every sum) took
// 5169 us; the F-cycle solve of that box 1091 -> 57 ms.  Above kBottomRegN
// nodes the values do not fit the registers of one workgroup.
constexpr int kBottomRegN = 256;
template <bool REG>
__global__ void __launch_bounds__(REG ? 512 : 1024)
    k_bottom_bicgstab(double* __restrict__ xg, const double* __restrict__ rhs, const double* __restrict__ vals,
                      const unsigned short* __restrict__ cols, const double* __restrict__ diag, int N, double omega,
                      int maxiter, double eps_rel, int nuf, int* __restrict__ status) {
    extern __shared__ double sm[];
    __shared__ double red[6][16];
    const int M = 3 * N;
    double *in = sm, *x = sm + M, *rh = sm + 2 * M, *p = sm + 3 * M, *v = sm + 4 * M;
    const int tid = threadIdx.x, node = tid >> 1, half = tid & 1, wave = tid >> 6, nw = blockDim.x >> 6;
    const bool on = node < N, own = on && half == 0;  // own: this thread keeps the node's entries of x, rh and in
    const long plane = 2L * kRowHalf * N;
    const int at0 = 2 * (on ? node : 0) + half;
    // REG: the values and, two to a register, the columns' byte offsets in `in`
    double a[3][REG ? kRowHalf : 1];
    unsigned off[REG ? (kRowHalf + 1) / 2 : 1];
    if constexpr (REG) {
#pragma unroll
        for (int k = 0; k < kRowHalf; ++k) {
            const long at = (long)k * 2 * N + at0;
            const unsigned c = 8u * cols[at];
            if (k & 1) off[k / 2] |= c << 16;
            else off[k / 2] = c;
#pragma unroll
            for (int r = 0; r < 3; ++r) a[r][k] = vals[at + r * plane];
        }
    }
    // A chunk's operands are read ahead of the chunk before it (REG), no more of
    // them at once than the registers hold beside the values.
    constexpr int CH = 5, NCH = (kRowHalf + CH - 1) / CH;
    auto matvec = [&](double y[3]) {
        y[0] = y[1] = y[2] = 0.0;
        if constexpr (REG) {
            double xv[2][CH];
            // keeps the compiler from unpacking all the offsets once, into registers that are not there
#pragma unroll
            for (unsigned& o : off) asm("" : "+v"(o));
            auto load = [&](int ch) {
#pragma unroll
                for (int e = 0; e < CH; ++e) {
                    const int k = ch * CH + e;
                    if (k >= kRowHalf) break;
                    const unsigned o = (k & 1) ? off[k / 2] >> 16 : off[k / 2] & 0xffffu;
                    xv[ch & 1][e] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(in) + o);
                }
            };
            load(0);
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) {
                if (ch + 1 < NCH) load(ch + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < CH; ++e) {
                    if (ch * CH + e >= kRowHalf) break;
#pragma unroll
                    for (int r = 0; r < 3; ++r) y[r] += a[r][ch * CH + e] * xv[ch & 1][e];
                }
            }
        } else {
#pragma unroll 1
            for (int ch = 0; ch < NCH; ++ch) {
                double av[3][CH], xv[CH];
#pragma unroll
                for (int e = 0; e < CH; ++e) {
                    const int k = ch * CH + e;
                    const bool have = k < kRowHalf;
                    const long at = (long)(have ? k : 0) * 2 * N + at0;
                    xv[e] = in[cols[at]];
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        av[r][e] = vals[at + r * plane];
                        if (!have) av[r][e] = 0.0;
                    }
                }
#pragma unroll
                for (int e = 0; e < CH; ++e)
#pragma unroll
                    for (int r = 0; r < 3; ++r) y[r] += av[r][e] * xv[e];
            }
        }
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            y[r] += dpp_f64<0xB1>(y[r]);
            if (!on) y[r] = 0.0;
        }
    };
    auto put = [&](double* v, const double e[3]) {
        if (own) {
            v[node] = e[0];
            v[N + node] = e[1];
            v[2 * N + node] = e[2];
        }
    };
    // the waves' values in red[slot] folded after the caller's barrier
    auto fold = [&](int slot, bool mx) {
        double r = red[slot][0];
        for (int q = 1; q < nw; ++q) r = mx ? fmax(r, red[slot][q]) : r + red[slot][q];
        return r;
    };
    auto post = [&](int slot, double v) {
        if ((tid & 63) == 0) red[slot][wave] = v;
    };
    double r[3], t[3];
    const double zero[3] = {0, 0, 0};
    double lm = 0.0, l1 = 0.0, l2 = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        r[c] = on ? rhs[c * N + node] / diag[c * N + node] : 0.0;  // x = 0
        lm = fmax(lm, fabs(r[c]));
        if (own) l1 += r[c] * r[c];
    }
    put(rh, r);
    put(x, zero);
    post(0, wave_all<true>(lm));
    post(1, wave_all<false>(l1));
    __syncthreads();
    const double rnorm0 = fold(0, true);
    double rho = fold(1, false);
    double rnorm = rnorm0, rho_1 = 0.0, alpha = 0.0, omg = 0.0;
    int ret = 0;
    if (rnorm0 != 0.0) {
        for (int iter = 1; iter <= maxiter; ++iter) {
            if (rho == 0.0) { ret = 1; break; }
            const double beta = iter == 1 ? 0.0 : (rho / rho_1) * (alpha / omg);
            if (own)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int q = c * N + node;
                    const double e = iter == 1 ? r[c] : r[c] + beta * (p[q] + (-omg) * v[q]);
                    p[q] = e;
                    in[q] = e;
                }
            __syncthreads();
            matvec(t);
            put(v, t);
            l1 = 0.0;
            if (own) l1 = rh[node] * t[0] + rh[N + node] * t[1] + rh[2 * N + node] * t[2];
            post(2, wave_all<false>(l1));
            __syncthreads();
            const double rhTv = fold(2, false);
            if (rhTv != 0.0) alpha = rho / rhTv;
            else { ret = 2; break; }
            lm = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (own) x[c * N + node] += alpha * p[c * N + node];
                r[c] += (-alpha) * t[c];  // s
                lm = fmax(lm, fabs(r[c]));
            }
            put(in, r);
            post(3, wave_all<true>(lm));
            __syncthreads();
            matvec(t);
            l1 = l2 = 0.0;
            if (own)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    l1 += t[c] * t[c];
                    l2 += t[c] * r[c];
                }
            post(4, wave_all<false>(l1));
            post(5, wave_all<false>(l2));
            __syncthreads();
            rnorm = fold(3, true);
            if (rnorm < eps_rel * rnorm0) break;
            const double tt = fold(4, false), ts = fold(5, false);
            if (tt != 0.0) omg = ts / tt;
            else { ret = 3; break; }
            lm = l1 = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (own) x[c * N + node] += omg * r[c];
                r[c] += (-omg) * t[c];
                lm = fmax(lm, fabs(r[c]));
            }
            if (own) l1 = rh[node] * r[0] + rh[N + node] * r[1] + rh[2 * N + node] * r[2];
            post(0, wave_all<true>(lm));
            post(1, wave_all<false>(l1));
            __syncthreads();
            rnorm = fold(0, true);
            if (rnorm < eps_rel * rnorm0) break;
            if (omg == 0.0) { ret = 4; break; }
            rho_1 = rho;
            rho = fold(1, false);
        }
        if (ret == 0 && rnorm > eps_rel * rnorm0) ret = 8;
        // x is kept only when it reduced the residual and the solve ended well
        if (!(ret == 0 && rnorm < rnorm0)) put(x, zero);
        // nuf Fsmooth calls after a failure, from x = 0; r holds x here
        const int nsm = ret == 0 ? 0 : nuf;
        if (nsm > 0) {
            double bd[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                r[c] = 0.0;
                bd[c] = on ? rhs[c * N + node] / diag[c * N + node] : 0.0;
            }
            for (int sw = 0; sw < 2 * nsm; ++sw) {
                __syncthreads();
                put(in, r);
                __syncthreads();
                matvec(t);
#pragma unroll
                for (int c = 0; c < 3; ++c) r[c] = (1.0 - omega) * r[c] + omega * (bd[c] - (t[c] - r[c]));
            }
            put(x, r);
        }
    }
    if (own)
        for (int c = 0; c < 3; ++c) xg[c * N + node] = x[c * N + node];
    if (tid == 0) status[0] = ret;
}

}  // namespace ael
