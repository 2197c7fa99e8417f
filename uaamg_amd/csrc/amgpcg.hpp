// amgpcg.hpp -- the standalone Ax=b amgpcg entry point on the GPU.
//
// Semantics of the reference's standalone amgpcg (test/solver/test_amgpcg.cpp:6-70
// with test/test_common.h:7-97): N x N node-centred Dirichlet Poisson
// (h = 1/(N+1), ghost = 0), row-major v[i*(N+2)+j]; levels N, N/2, ... down to
// <= 3; V-cycle: 2 RBGS sweeps, residual, restrict 0.25*sum(2x2) into a coarse
// grid of size N/2 made even (read back with that grid's own row stride, so an
// odd level gets a zero last row/column), recurse, prolong x1.0, 2 RBGS sweeps;
// 20 sweeps on the coarsest.  RBGS: first (i+j) odd, then (i+j) even,
// x += h^2/4 (b - A x).  PCG with absolute tolerance, out_iters = k+1.
#pragma once
#include <functional>
#include "amgpcg_plan.hpp"
#include "engine.hpp"

namespace uaamg {

template <typename T>
__global__ void k_cast_all_ag(const double* __restrict__ src, T* __restrict__ dst, long n, int N) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    long i = t / (N + 2), j = t % (N + 2);
    dst[t] = (i >= 1 && i <= N && j >= 1 && j <= N) ? (T)src[t] : T(0);
}
template <typename T>
__global__ void k_cast_all_ag_out(const T* __restrict__ src, double* __restrict__ dst, long n) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dst[t] = (double)src[t];
}

template <typename T>
__device__ __forceinline__ T ag_lap(T xc, T up, T dn, T xr, T xl, T inv_h2) {
    // (i+1, i-1, j+1, j-1) in the order the reference subtracts them
    return (T(4) * xc - up - dn - xr - xl) * inv_h2;
}

// Scalars of one solve.  rs[k & 1] is iteration k's r.z, written by its
// operator launch and read by later ones; done / iter are written by the tail.
struct AgCtrl {
    double rs[2];
    int done, iter;
};

// sum of nb partials, the same value in every thread (fixed order)
__device__ __forceinline__ double ag_total(const double* partials, int nb) {
    __shared__ double all;
    double v[1];
    reduce_partials<1>(partials, nb, v);
    if (lin_thread() == 0) all = v[0];
    __syncthreads();
    return all;
}

// n partials in fixed shares to AG_FOLD sums, one workgroup each (ag_plan).
// With every workgroup adding all partials, an iteration of a large solve
// went mostly into that (us an iteration, FP64: N = 1500 158 -> 150, 2048 384 -> 329,
// 4096 1306 -> 805, 6144 4378 -> 1685; N = 1024 99, with the fold 111).
__global__ __launch_bounds__(256) void k_ag_fold(const double* __restrict__ in, int n, double* __restrict__ out, const int* done) {
    if (*done) return;
    const int len = (n + AG_FOLD - 1) / AG_FOLD, beg = (int)blockIdx.x * len, end = min(n, beg + len);
    double v[1] = {0.0};
    for (int k = beg + (int)threadIdx.x; k < end; k += 256) v[0] += in[k];
    block_sum<1>(v);
    if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

// ---- tile kernels: one launch down and one up per level ----
//
// A workgroup owns AT_X x AT_Y cells of a level plus a halo of AT_H cells;
// a thread owns two neighbouring cells of a row (one of each colour) with
// their b in registers.  x lives in LDS, the left and the right cells of the
// pairs in separate arrays, so a colour pass reads three neighbours at unit
// stride (the fourth is the pair's other cell) and writes one value.  A pass
// spoils one more ring of the region from its edge; going down x starts at 0,
// so the first pass spoils none and the residual's ring is covered too.
// These levels are latency-bound (a 256^2 FP64 level is 0.5 MB): with every
// colour pass, restriction and prolongation a launch of its own an N = 256
// FP64 solve took 6.6 ms with the GPU busy for 12 % of it, now 1.1 ms.
constexpr int AT_H = 4, AT_THREADS = 512;
constexpr int AT_RX = AT_X + 2 * AT_H, AT_RY = AT_Y + 2 * AT_H, AT_HX = AT_RX / 2, AT_SX = AT_HX + 2;
constexpr int AT_N = AT_SX * (AT_RY + 2);   // one side's LDS array: the pairs and a ring that stays 0
static_assert(AT_HX * AT_RY <= AT_THREADS && AT_H % 2 == 0 && AT_X % 2 == 0 && AT_Y % 2 == 0, "pairs are the coarse cells' children");

template <typename T>
struct AgPair {
    int gi, gj, e;       // row, column of the left cell (1-based level coordinates), LDS index
    bool own, in0, in1;  // in the tile (not the halo); the cells lie in the level
    bool left_odd;       // the left cell has the odd colour
    long id;
    T x0, x1, b0, b1;
    __device__ __forceinline__ void place(int N) {
        const int t = (int)threadIdx.x, rj = t / AT_HX, hx = t % AT_HX;
        const bool live = t < AT_HX * AT_RY;
        gi = 1 + (int)blockIdx.y * AT_Y - AT_H + rj;
        gj = 1 + (int)blockIdx.x * AT_X - AT_H + 2 * hx;
        e = live ? (rj + 1) * AT_SX + hx + 1 : 0;
        const bool row = live && gi >= 1 && gi <= N;
        in0 = row && gj >= 1 && gj <= N;
        in1 = row && gj + 1 >= 1 && gj + 1 <= N;
        own = rj >= AT_H && rj < AT_H + AT_Y && 2 * hx >= AT_H && 2 * hx < AT_H + AT_X;
        left_odd = ((gi + gj) & 1) != 0;
        id = (long)gi * (N + 2) + gj;
        x0 = x1 = b0 = b1 = T(0);
    }
    // one colour pass
    __device__ __forceinline__ void pass(T* X, bool odd, T inv_h2, T inv_diag) {
        const bool left = left_odd == odd;
        T* A = left ? X : X + AT_N;
        const T* O = left ? X + AT_N : X;
        if (left ? in0 : in1) {
            const T xc = left ? x0 : x1;
            const T xl = left ? O[e - 1] : x0, xr = left ? x1 : O[e + 1];
            const T v = xc + inv_diag * ((left ? b0 : b1) - ag_lap(xc, A[e + AT_SX], A[e - AT_SX], xr, xl, inv_h2));
            A[e] = v;
            if (left) x0 = v;
            else x1 = v;
        }
        __syncthreads();
    }
    __device__ __forceinline__ void sweeps(T* X, T inv_h2, T inv_diag) {
        pass(X, true, inv_h2, inv_diag);
        pass(X, false, inv_h2, inv_diag);
        pass(X, true, inv_h2, inv_diag);
        pass(X, false, inv_h2, inv_diag);
    }
};

// What the level-0 down launch does of the CG update first: alpha, x += alpha p
// and r_new = r - alpha Ap (r_new to the other r buffer: other workgroups
// still read r on their halo), r.r partials.
template <typename T>
struct AgUpdate {
    T* x; const T* p; const T* r; const T* Ap; T* r_new;
    const double* pAp; int npAp;
    double* rr;          // nullptr: no update, b is r_new as it stands
    const AgCtrl* c; int slot;
};

// Down: x = 0, two sweeps, x written; restriction of the residual,
// bc(ic, jc) = 0.25 * the sum of the 2x2 children's for ic, jc <= Nc, else 0.
template <typename T, bool UPD>
__global__ __launch_bounds__(AT_THREADS) void k_ag_down(T* __restrict__ x, const T* __restrict__ b, int N, T inv_h2, T inv_diag,
                                                        T* __restrict__ bc, int Nb, int Nc, AgUpdate<T> u, const int* done) {
    if (*done) return;
    __shared__ T X[2 * AT_N];
    AgPair<T> c;
    c.place(N);
    for (int k = threadIdx.x; k < 2 * AT_N; k += AT_THREADS) X[k] = T(0);
    if constexpr (UPD) {
        T r0 = T(0), r1 = T(0), a0 = T(0), a1 = T(0), p0 = T(0), p1 = T(0), y0 = T(0), y1 = T(0);
        if (c.in0) { r0 = u.r[c.id]; a0 = u.Ap[c.id]; }
        if (c.in1) { r1 = u.r[c.id + 1]; a1 = u.Ap[c.id + 1]; }
        if (c.own && c.in0) { p0 = u.p[c.id]; y0 = u.x[c.id]; }
        if (c.own && c.in1) { p1 = u.p[c.id + 1]; y1 = u.x[c.id + 1]; }
        const double alpha = u.c->rs[u.slot] / ag_total(u.pAp, u.npAp);
        c.b0 = c.in0 ? (T)((double)r0 + -alpha * (double)a0) : T(0);
        c.b1 = c.in1 ? (T)((double)r1 + -alpha * (double)a1) : T(0);
        double v[1] = {0.0};
        if (c.own && c.in0) {
            u.x[c.id] = (T)((double)y0 + alpha * (double)p0);
            u.r_new[c.id] = c.b0;
            v[0] += (double)c.b0 * (double)c.b0;
        }
        if (c.own && c.in1) {
            u.x[c.id + 1] = (T)((double)y1 + alpha * (double)p1);
            u.r_new[c.id + 1] = c.b1;
            v[0] += (double)c.b1 * (double)c.b1;
        }
        block_store<1>(v, u.rr);
    } else {
        if (c.in0) c.b0 = b[c.id];
        if (c.in1) c.b1 = b[c.id + 1];
    }
    __syncthreads();
    c.sweeps(X, inv_h2, inv_diag);
    if (c.own && c.in0) x[c.id] = c.x0;
    if (c.own && c.in1) x[c.id + 1] = c.x1;
    // residuals of the pair, then of the pair below it, in LDS
    T* XL = X;
    T* XR = X + AT_N;
    T r0 = T(0), r1 = T(0);
    if (c.own) {
        r0 = c.b0 - ag_lap(c.x0, XL[c.e + AT_SX], XL[c.e - AT_SX], c.x1, XR[c.e - 1], inv_h2);
        r1 = c.b1 - ag_lap(c.x1, XR[c.e + AT_SX], XR[c.e - AT_SX], XL[c.e + 1], c.x0, inv_h2);
    }
    __syncthreads();
    if (c.own) { XL[c.e] = r0; XR[c.e] = r1; }
    __syncthreads();
    if (c.own && (c.gi & 1)) {
        const int ic = (c.gi + 1) >> 1, jc = (c.gj + 1) >> 1;
        if (ic <= Nb && jc <= Nb)
            bc[(long)ic * (Nb + 2) + jc] = (ic <= Nc && jc <= Nc) ? T(0.25) * (r0 + XL[c.e + AT_SX] + r1 + XR[c.e + AT_SX]) : T(0);
    }
}

// Up: x = xd + the parent's x (xc, level size Nb), two sweeps; written to xo
// (other workgroups still read xd on their halo).  DOT: partials of b.x.
template <typename T, bool DOT>
__global__ __launch_bounds__(AT_THREADS) void k_ag_up(const T* __restrict__ xd, T* __restrict__ xo, const T* __restrict__ b, int N,
                                                      T inv_h2, T inv_diag, const T* __restrict__ xc, int Nb, double* partials,
                                                      const int* done) {
    if (*done) return;
    __shared__ T X[2 * AT_N];
    AgPair<T> c;
    c.place(N);
    const int ic = (c.gi + 1) >> 1, jc = (c.gj + 1) >> 1;
    T cv = T(0);
    if (c.in0) { c.b0 = b[c.id]; c.x0 = xd[c.id]; }
    if (c.in1) { c.b1 = b[c.id + 1]; c.x1 = xd[c.id + 1]; }
    if (c.in0 && ic <= Nb && jc <= Nb) cv = xc[(long)ic * (Nb + 2) + jc];   // in0: gj is odd, so in1 alone cannot be
    for (int k = threadIdx.x; k < 2 * AT_N; k += AT_THREADS) X[k] = T(0);
    __syncthreads();
    if (c.in0) X[c.e] = c.x0 = c.x0 + cv;
    if (c.in1) X[AT_N + c.e] = c.x1 = c.x1 + cv;
    __syncthreads();
    c.sweeps(X, inv_h2, inv_diag);
    if (c.own && c.in0) xo[c.id] = c.x0;
    if (c.own && c.in1) xo[c.id + 1] = c.x1;
    if constexpr (DOT) {
        double v[1] = {0.0};
        if (c.own && c.in0) v[0] += (double)c.b0 * (double)c.x0;
        if (c.own && c.in1) v[0] += (double)c.b1 * (double)c.x1;
        block_store<1>(v, partials);
    }
}

// ---- the levels of at most AG_TAIL cells a side, in one workgroup ----
constexpr int AG_TAIL_THREADS = 1024, AG_TAIL_MAXL = 8;
constexpr int AG_TAIL_CELLS = 6016;   // >= the padded cells of 64, 32, 16, 8, 4, 2

struct AgTail {
    int nl;                           // levels here; the last is the coarsest (side <= 3)
    int n[AG_TAIL_MAXL], nc[AG_TAIL_MAXL], off[AG_TAIL_MAXL];
    const double* rr; int nrr;        // this iteration's r.r partials (nullptr: no convergence test)
    double tol; int iter;
    double* dot;                      // where b.x of the first level goes (nullptr: not wanted)
    AgCtrl* c;
};

// The coarsest level's sweeps (side S, at most 3) in one thread's registers:
// 2 x 20 passes over at most nine cells, each pass a short dependent chain.
template <typename T, int S>
__device__ __forceinline__ void ag_coarsest(T* X, const T* B, T inv_h2, T inv_diag, int sweeps) {
    constexpr int R = S + 2;
    T x[R * R], b[R * R];
#pragma unroll
    for (int k = 0; k < R * R; k++) { x[k] = X[k]; b[k] = B[k]; }
    for (int s = 0; s < sweeps; s++)
#pragma unroll
        for (int odd = 1; odd >= 0; odd--)
#pragma unroll
            for (int i = 1; i <= S; i++)
#pragma unroll
                for (int j = 1; j <= S; j++)
                    if (((i + j) & 1) == odd) {
                        const int e = i * R + j;
                        x[e] = x[e] + inv_diag * (b[e] - ag_lap(x[e], x[e + R], x[e - R], x[e + 1], x[e - 1], inv_h2));
                    }
#pragma unroll
    for (int k = 0; k < R * R; k++) X[k] = x[k];
}

template <typename T>
__global__ __launch_bounds__(AG_TAIL_THREADS) void k_ag_tail(AgTail A, const T* __restrict__ b, T* __restrict__ x) {
    if (A.c->done) return;
    __shared__ T X[AG_TAIL_CELLS];
    __shared__ T B[AG_TAIL_CELLS];
    __shared__ int stop;
    const int tid = (int)threadIdx.x;
    const int n0 = A.n[0], N0 = (n0 + 2) * (n0 + 2);
    for (int e = tid; e < AG_TAIL_CELLS; e += AG_TAIL_THREADS) {
        X[e] = T(0);
        T v = T(0);
        if (e < N0) {
            const int i = e / (n0 + 2), j = e % (n0 + 2);
            if (i >= 1 && i <= n0 && j >= 1 && j <= n0) v = b[e];
        }
        B[e] = v;
    }
    if (A.rr) {   // sqrt(r.r) < tol after this iteration's update: the solve ends before the V-cycle
        double v[1];
        reduce_partials<1>(A.rr, A.nrr, v);
        if (tid == 0) {
            stop = sqrt(v[0]) < A.tol;
            if (stop) { A.c->iter = A.iter; A.c->done = 1; }
        }
        __syncthreads();
        if (stop) return;
    }
    __syncthreads();
    auto ih2 = [](int n) { const double h = 1.0 / (n + 1); return (T)(1.0 / (h * h)); };
    auto idg = [](int n) { const double h = 1.0 / (n + 1); return (T)(h * h / 4.0); };
    // levels of at most 8 a side (32 cells of a colour) run on wave 0 alone:
    // the LDS accesses of one wave complete in order, so no barrier
    auto sync = [&](bool wave) {
        if (wave) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            __syncthreads();
        }
    };
    auto smooth = [&](int l, bool wave) {
        const int n = A.n[l], R = n + 2, hx = (n + 1) / 2, nt = wave ? 64 : AG_TAIL_THREADS;
        T* Xl = X + A.off[l];
        const T* Bl = B + A.off[l];
        const T h2 = ih2(n), dg = idg(n);
        for (int q = 0; q < 4; q++) {
            const int odd = 1 - (q & 1);
            for (int k = tid; k < n * hx; k += nt) {
                const int i = 1 + k / hx, j = 1 + ((odd + 1 + i) & 1) + 2 * (k % hx);
                if (j > n) continue;
                const int e = i * R + j;
                Xl[e] = Xl[e] + dg * (Bl[e] - ag_lap(Xl[e], Xl[e + R], Xl[e - R], Xl[e + 1], Xl[e - 1], h2));
            }
            sync(wave);
        }
    };
    auto down = [&](int l, bool wave) {
        smooth(l, wave);
        const int n = A.n[l], R = n + 2, nb = A.n[l + 1], nc = A.nc[l], nt = wave ? 64 : AG_TAIL_THREADS;
        const T* Xl = X + A.off[l];
        const T* Bl = B + A.off[l];
        const T h2 = ih2(n);
        auto res = [&](int e) { return Bl[e] - ag_lap(Xl[e], Xl[e + R], Xl[e - R], Xl[e + 1], Xl[e - 1], h2); };
        for (int k = tid; k < nb * nb; k += nt) {
            const int ic = 1 + k / nb, jc = 1 + k % nb;
            T v = T(0);
            if (ic <= nc && jc <= nc) {
                const int e = (2 * ic - 1) * R + 2 * jc - 1;
                v = T(0.25) * (res(e) + res(e + R) + res(e + 1) + res(e + R + 1));
            }
            B[A.off[l + 1] + ic * (nb + 2) + jc] = v;
        }
        sync(wave);
    };
    auto up = [&](int l, bool wave) {
        const int n = A.n[l], R = n + 2, nb = A.n[l + 1], nt = wave ? 64 : AG_TAIL_THREADS;
        T* Xl = X + A.off[l];
        const T* Xc = X + A.off[l + 1];
        for (int k = tid; k < n * n; k += nt) {
            const int i = 1 + k / n, j = 1 + k % n, ic = (i + 1) >> 1, jc = (j + 1) >> 1;
            const T c = (ic <= nb && jc <= nb) ? Xc[ic * (nb + 2) + jc] : T(0);
            Xl[i * R + j] = Xl[i * R + j] + c;
        }
        sync(wave);
        smooth(l, wave);
    };
    const int last = A.nl - 1;
    int lw = 0;   // first level that wave 0 runs alone
    while (lw < last && A.n[lw] > 8) lw++;
    for (int l = 0; l < lw; l++) down(l, false);
    if (tid < 64) {
        for (int l = lw; l < last; l++) down(l, true);
        const int n = A.n[last];
        if (tid == 0) {
            if (n == 3) ag_coarsest<T, 3>(X + A.off[last], B + A.off[last], ih2(3), idg(3), 20);
            else ag_coarsest<T, 2>(X + A.off[last], B + A.off[last], ih2(2), idg(2), 20);
        }
        sync(true);
        for (int l = last - 1; l >= lw; l--) up(l, true);
    }
    __syncthreads();
    for (int l = lw - 1; l >= 0; l--) up(l, false);
    double v[1] = {0.0};
    for (int k = tid; k < n0 * n0; k += AG_TAIL_THREADS) {
        const int e = (1 + k / n0) * (n0 + 2) + 1 + k % n0;
        x[e] = X[e];
        v[0] += (double)B[e] * (double)X[e];
    }
    if (A.dot) {
        block_sum<1>(v);
        if (tid == 0) *A.dot = v[0];
    }
}

// ---- CG passes ----

// p = z + beta p (written to the other p buffer: neighbours still read p) and
// Ap, p.Ap partials.  beta = r.z / the last iteration's (k = 0: 0, p is 0).
constexpr int AP_ROWS = 4;
template <typename T>
__global__ __launch_bounds__(AP_X * AP_Y / AP_ROWS) void k_ag_pmv(const T* __restrict__ z, const T* __restrict__ p, T* __restrict__ pn,
                                                                  T* __restrict__ Ap, int N, T inv_h2, const double* rz, int nrz,
                                                                  AgCtrl* c, int k, double* partials) {
    if (c->done) return;
    const double rs = ag_total(rz, nrz);
    const double beta = k ? rs / c->rs[(k - 1) & 1] : 0.0;
    if (lin_block() == 0 && lin_thread() == 0) c->rs[k & 1] = rs;
    const long s = N + 2;
    auto at = [&](long id) { return (T)((double)z[id] + beta * (double)p[id]); };
    double v[1] = {0.0};
    const int j = 1 + (int)blockIdx.x * AP_X + (int)threadIdx.x;
#pragma unroll
    for (int q = 0; q < AP_ROWS; q++) {
        const int i = 1 + (int)blockIdx.y * AP_Y + q * (AP_Y / AP_ROWS) + (int)threadIdx.y;
        if (i > N || j > N) continue;
        const long id = (long)i * s + j;
        const T pc = at(id);
        const T a = ag_lap(pc, at(id + s), at(id - s), at(id + 1), at(id - 1), inv_h2);
        pn[id] = pc;
        Ap[id] = a;
        v[0] += (double)pc * (double)a;
    }
    block_store<1>(v, partials);
}

// x += alpha p, r -= alpha Ap, r.r partials: the CG update where level 0 is in the tail
template <typename T>
__global__ __launch_bounds__(256) void k_ag_update(AgUpdate<T> u, int N, const int* done) {
    if (*done) return;
    const double alpha = u.c->rs[u.slot] / ag_total(u.pAp, u.npAp);
    double v[1] = {0.0};
    for (int t = (int)blockIdx.x * 256 + (int)threadIdx.x; t < N * N; t += (int)gridDim.x * 256) {
        const long id = (long)(1 + t / N) * (N + 2) + 1 + t % N;
        const T r = (T)((double)u.r[id] + -alpha * (double)u.Ap[id]);
        u.x[id] = (T)((double)u.x[id] + alpha * (double)u.p[id]);
        u.r_new[id] = r;
        v[0] += (double)r * (double)r;
    }
    block_store<1>(v, u.rr);
}

// Level sizes of the amgpcg hierarchy: N, N/2, ... down to <= 3 (test_amgpcg.cpp:66-71)
inline std::vector<int> amgpcg_levels(int N) {
    std::vector<int> lv;
    for (int n = N; n >= 2;) { lv.push_back(n); if (n <= 3) break; n = n / 2; if (n < 2) n = 2; }
    return lv;
}

// Device buffers of one amgpcg solve, carved in order from one arena (each
// start 256-byte aligned): per level x and b, then x, r, z, p, Ap, the dot
// partials and the scalar slot.  (Level 0's x and b hold the second r and p
// buffers; the other tile levels' second x lies in Ap, which nothing reads
// between the down leg and the next operator pass.)
constexpr size_t kAgAlign = 256;
inline size_t ag_round(size_t b) { return (b + kAgAlign - 1) / kAgAlign * kAgAlign; }
inline dim3 ag_tiles(int n) { return dim3((n + AT_X - 1) / AT_X, (n + AT_Y - 1) / AT_Y); }

template <typename T>
size_t amgpcg_arena_bytes(int N) {
    size_t bytes = 0;
    for (int n : amgpcg_levels(N)) bytes += 2 * ag_round((size_t)(n + 2) * (n + 2) * sizeof(T));
    const size_t NN = (size_t)(N + 2) * (N + 2);
    bytes += 5 * ag_round(NN * sizeof(T));
    bytes += ag_round(ag_partials_room(N) * sizeof(double)) + ag_round(64);
    return bytes;
}

// The solve on device arrays: b_dev (FP64, (N+2)^2 row-major, interior read)
// and x_dev (FP64, (N+2)^2, written whole).  `arena` holds at least
// amgpcg_arena_bytes<T>(N) bytes; it is cleared here.  The CG scalars stay on
// the device (six launches per iteration at N = 256); the host reads the done
// flag (hscal: 64 bytes of host memory, pinned or not) after every
// AG_CHECK iterations, and iterations queued past the stop return at once.
constexpr int AG_CHECK = 4;
template <typename T>
int amgpcg_core(int N, const double* b_dev, double* x_dev, int max_iter, double tol, int* iters,
                unsigned char* arena, size_t arena_bytes, hipStream_t s, double* hscal) {
    const std::vector<int> lv = amgpcg_levels(N);
    const int nl = (int)lv.size();
    const size_t need = amgpcg_arena_bytes<T>(N);
    if (need > arena_bytes) throw HipError{hipErrorInvalidValue, "amgpcg arena too small"};
    HIPCHK(hipMemsetAsync(arena, 0, need, s));
    size_t used = 0;
    auto take = [&](size_t bytes) {
        void* p = arena + used;
        used += ag_round(bytes);
        return p;
    };
    const size_t NN = (size_t)(N + 2) * (N + 2);
    std::vector<T*> X(nl), B(nl), X2(nl, nullptr);
    for (int l = 0; l < nl; l++) {
        size_t n2 = (size_t)(lv[l] + 2) * (lv[l] + 2);
        X[l] = (T*)take(n2 * sizeof(T)); B[l] = (T*)take(n2 * sizeof(T));
    }
    T *x = (T*)take(NN * sizeof(T)), *r = (T*)take(NN * sizeof(T)), *z = (T*)take(NN * sizeof(T));
    T *p = (T*)take(NN * sizeof(T)), *Ap = (T*)take(NN * sizeof(T));
    T* rb[2] = {r, B[0]};
    T* pb[2] = {p, X[0]};
    const dim3 mgrid((N + AP_X - 1) / AP_X, (N + AP_Y - 1) / AP_Y), mblk(AP_X, AP_Y / AP_ROWS);
    const AgPlan plan = ag_plan(N);
    const int nm = plan.nm, nu = plan.nu;
    if (plan.doubles > ag_partials_room(N)) throw HipError{hipErrorInvalidValue, "amgpcg: partial sums do not fit"};
    double* part_m = (double*)take(ag_partials_room(N) * sizeof(double));
    AgCtrl* ctrl = (AgCtrl*)take(64);
    double* part_z = part_m + nm;    // r.r partials first, then r.z (the tail has read the former before the last up launch)
    // what the consumers add
    double* sum_m = plan.fold ? part_z + nu : part_m;
    double* sum_z = plan.fold ? sum_m + AG_FOLD : part_z;
    auto fold = [&](const double* part, int n, double* sum) {
        if (plan.fold) k_ag_fold<<<AG_FOLD, 256, 0, s>>>(part, n, sum, &ctrl->done);
    };

    int lt = 0;                      // first level of the tail
    while (lv[lt] > AG_TAIL) lt++;
    const dim3 tgrid = ag_tiles(N);
    AgTail tail{};
    tail.nl = nl - lt;
    for (int l = lt, off = 0; l < nl; l++) {
        tail.n[l - lt] = lv[l];
        tail.off[l - lt] = off;
        off += (lv[l] + 2) * (lv[l] + 2);
    }
    auto nc_of = [&](int l) { int nc = lv[l] / 2; if (nc < 2) nc = 2; if (nc % 2 != 0 && nc > 2) nc--; return nc; };
    for (int l = lt; l < nl - 1; l++) tail.nc[l - lt] = nc_of(l);
    tail.tol = tol;
    tail.c = ctrl;
    {
        size_t o = 0;
        for (int l = 1; l < lt; l++) { X2[l] = Ap + o; o += ag_round((size_t)(lv[l] + 2) * (lv[l] + 2) * sizeof(T)) / sizeof(T); }
    }

    k_cast_all_ag<T><<<(unsigned)((NN + 255) / 256), 256, 0, s>>>(b_dev, r, (long)NN, N);

    auto h_of = [](int n) { return 1.0 / (n + 1); };
    auto ih2 = [&](int n) { double h = h_of(n); return (T)(1.0 / (h * h)); };
    auto idg = [&](int n) { double h = h_of(n); return (T)(h * h / 4.0); };
    // z = M^-1 of rb[(k + 1) & 1] and its r.z partials; k >= 0: iteration k's
    // CG update and convergence test with it (k = -1: neither).  The p buffer
    // that iteration k + 1 writes holds level 0's x between the legs.
    auto precond = [&](int k) {
        const T* rr = rb[(k + 1) & 1];
        T* zd = pb[k & 1];
        AgUpdate<T> u{};
        if (k >= 0) u = AgUpdate<T>{x, pb[(k + 1) & 1], rb[k & 1], Ap, rb[(k + 1) & 1], sum_m, plan.sum_m, part_z, ctrl, k & 1};
        for (int l = 0; l < lt; l++) {
            T* xl = l ? X[l] : zd;
            const T* bl = l ? B[l] : rr;
            if (l == 0 && k >= 0)
                k_ag_down<T, true><<<tgrid, AT_THREADS, 0, s>>>(xl, bl, lv[l], ih2(lv[l]), idg(lv[l]), B[l + 1], lv[l + 1], nc_of(l), u, &ctrl->done);
            else
                k_ag_down<T, false><<<ag_tiles(lv[l]), AT_THREADS, 0, s>>>(xl, bl, lv[l], ih2(lv[l]), idg(lv[l]), B[l + 1], lv[l + 1], nc_of(l), u, &ctrl->done);
        }
        if (lt == 0 && k >= 0) k_ag_update<T><<<nu, 256, 0, s>>>(u, N, &ctrl->done);
        if (k >= 0) fold(part_z, nu, sum_z);
        tail.rr = k >= 0 ? sum_z : nullptr;
        tail.nrr = plan.fold ? AG_FOLD : nu;
        tail.iter = k + 1;
        tail.dot = lt == 0 ? part_z : nullptr;
        k_ag_tail<T><<<1, AG_TAIL_THREADS, 0, s>>>(tail, lt ? B[lt] : rr, lt ? X[lt] : z);
        for (int l = lt - 1; l >= 0; l--) {
            const T* xc = l + 1 < lt ? X2[l + 1] : X[l + 1];
            if (l == 0)
                k_ag_up<T, true><<<tgrid, AT_THREADS, 0, s>>>(zd, z, rr, N, ih2(N), idg(N), xc, lv[1], part_z, &ctrl->done);
            else
                k_ag_up<T, false><<<ag_tiles(lv[l]), AT_THREADS, 0, s>>>(X[l], X2[l], B[l], lv[l], ih2(lv[l]), idg(lv[l]), xc, lv[l + 1], nullptr, &ctrl->done);
        }
        fold(part_z, nu, sum_z);
    };
    precond(-1);
    int it_out = max_iter;
    for (int k = 0; k < max_iter;) {
        const int k1 = std::min(max_iter, k + AG_CHECK);
        for (; k < k1; k++) {
            k_ag_pmv<T><<<mgrid, mblk, 0, s>>>(z, pb[k & 1], pb[(k + 1) & 1], Ap, N, ih2(N), sum_z, plan.sum_z, ctrl, k, part_m);
            fold(part_m, nm, sum_m);
            precond(k);
        }
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(hscal, ctrl, sizeof(AgCtrl), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        AgCtrl hc;
        std::memcpy(&hc, hscal, sizeof(hc));
        if (hc.done) { it_out = hc.iter; break; }
    }
    HIPCHK(hipGetLastError());
    k_cast_all_ag_out<T><<<(unsigned)((NN + 255) / 256), 256, 0, s>>>(x, x_dev, (long)NN);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s));
    *iters = it_out;
    return UAAMG_OK;
}

// Host arrays in and out: the arena and a b/x staging array are allocated
// per call on a stream of its own.
template <typename T>
int amgpcg_run(int N, const double* b_host, double* x_host, int max_iter, double tol, int* iters) {
    hipStream_t s;
    HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    std::vector<void*> allocs;
    auto dal = [&](size_t bytes) {
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, bytes);
        if (e != hipSuccess) throw HipError{e, "hipMalloc"};
        allocs.push_back(p);
        return p;
    };
    struct Cleanup {
        std::vector<void*>& a; hipStream_t s;
        ~Cleanup() { (void)hipStreamSynchronize(s); for (void* p : a) (void)hipFree(p); (void)hipStreamDestroy(s); }
    } cleanup{allocs, s};
    const size_t NN = (size_t)(N + 2) * (N + 2);
    const size_t ab = amgpcg_arena_bytes<T>(N);
    unsigned char* arena = (unsigned char*)dal(ab);
    double* bd = (double*)dal(NN * sizeof(double));
    double* hscal = nullptr;
    HIPCHK(hipHostMalloc((void**)&hscal, 64, hipHostMallocDefault));
    struct HostFree { double* p; ~HostFree() { if (p) (void)hipHostFree(p); } } hf{hscal};
    HIPCHK(hipMemcpyAsync(bd, b_host, NN * sizeof(double), hipMemcpyHostToDevice, s));
    // bd holds b until the core has cast it into r, then receives x
    amgpcg_core<T>(N, bd, bd, max_iter, tol, iters, arena, ab, s, hscal);
    HIPCHK(hipMemcpyAsync(x_host, bd, NN * sizeof(double), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    return UAAMG_OK;
}

}  // namespace uaamg
