// kernels_tail.hpp -- the small coarse levels of the V-cycle in one
// workgroup.
//
// Below a few thousand cells a level is latency-bound: each separate launch
// costs more than its arithmetic.  k_tail runs the whole lower part of the
// V(1,1) cycle -- forward sweep, residual restriction, the coarsest
// 10 x (forward + reverse) sweeps, prolongation and reverse sweep for every
// level from `first` down to the coarsest -- in one 1024-thread workgroup
// with x, b and the residual of every tail level in LDS and the stencil
// records of the cells a thread owns in registers.  Arithmetic and order are
// those of the per-pass kernels (k_smooth, k_restrict, k_prolong), i.e. of
// the reference smooth / restrictResidual / prolongateAdd
// (uaamg_preconditioner_3d.cpp:123-196); the FP32 form divides by the
// hardware reciprocal, as the march kernels do.
//
// A thread owns pairs of x-adjacent cells (i odd, i+1): one cell of each
// colour, so every RBGS pass keeps all lanes busy.
//
// One workgroup on one CU: the chain of dependent steps is what counts.
//   * Everything a pair needs is built at set-up (k_tail_records): couplings,
//     diagonal and 1 / diagonal by colour, and the pair's LDS index, its
//     parent's and its first child's (integer divisions by the level's sides
//     cost as much as the memory round trip).  Only existing pairs are loaded.
//   * The kernel arguments that the loads depend on come first in the block,
//     so one round trip of scalar loads starts all of them.
//   * x = 0 before the first pass of a level, so that pass is b / d of the
//     thread's own cell, in the step that restricts b: three barriers a level
//     down, three up.
//   * Levels of at most 64 pairs run in wave 0 alone, without barriers.
//   * The convergence test costs no barrier of its own.
// Measured against the form before (records of all 1024 threads loaded,
// indices by division, four barriers a level, division in the chain): 16^3 to
// 4^3 FP32 19.6 -> 15.9 us, 18 x 12 x 7 FP32
// 13.4 -> 9.0, 16 x 8 x 8 FP64 24.0 -> 12.2, 2D 32 x 16 FP64 15.2 -> 13.3, 12 2D
// grids of up to 5 levels 20.7 -> 16.3.  What is left is the 21 coarsest passes
// (a chain of LDS reads and additions) and one memory round trip.
#pragma once
#include "kernels_cg.hpp"

namespace uaamg {

constexpr int TAIL_THREADS = 1024;
constexpr int TAIL_MAXL = 5;      // tail levels (3D: 16^3..4^3 is 3; 2D: 64^2..4^2 is 5)
constexpr int TAIL_MAXP = 2;      // pairs per thread on the first tail level
constexpr int TAIL_LDS_BYTES = 96 * 1024;   // x, b of every tail level + one residual array
constexpr int TAIL_BMAX = 8;     // b elements per thread of the first tail level (padded cells <= 8192; FP64: 4, by the LDS)

// A pair's record: 16 values (d, 1/d, xp, xm, yp, ym, zp, zm, each of the even
// and the odd cell; 1/d = 0 where no pass updates the cell) and 4 indices, in
// 16-byte quads stored [level][quad][pair], a level's pairs padded to whole
// waves, so that every quad load of a wave is one contiguous 1 KiB read.
template <typename CT> struct TailRec;
template <> struct TailRec<float> { static constexpr int NV = 4, NQ = 5, PER = 4; using Q = float4; };
template <> struct TailRec<double> { static constexpr int NV = 8, NQ = 9, PER = 2; using Q = double2; };
__host__ __device__ constexpr int tail_rec_stride(int np) { return (np + 63) / 64 * 64; }
template <typename CT> constexpr long tail_rec_bytes(int np) { return (long)tail_rec_stride(np) * TailRec<CT>::NQ * 16; }   // of a level
// pairs of a level (D = 3: nz planes; 2D levels have nz = 1)
inline int tail_pairs(const Geo& g) { return ((g.nx + 1) / 2) * g.ny * g.nz; }

template <typename C4>
struct TailArgs {
    // what the first loads depend on
    const void* rec;               // pair records (compute type)
    const void* b;                 // b of the first tail level (level storage type)
    void* x;                       // x of the first tail level (written at the end)
    const int* skip;               // stop flag (nullptr: never skip)
    // the convergence test of this iteration (k_fin_update), run before the
    // levels: r.r partials (k_tail: nullptr: no test here) and the scalars
    const double* rr;
    Ctrl* ctrl;
    int nrr;
    int nl;                        // levels in the tail; the last one is the coarsest
    int ro;                        // LDS offset of the residual scratch (behind x and b of every level)
    int N0;                        // padded cells of the first one
    int np[TAIL_MAXL];             // pairs per level (0 past nl)
    int rq[TAIL_MAXL];             // a level's first quad in rec
    int npass;                     // coarsest passes (2 * sweeps + 1)
    int xo[TAIL_MAXL], bo[TAIL_MAXL];   // LDS offsets (elements) of x and b per level
    Geo g[TAIL_MAXL];
    const C4* coef[TAIL_MAXL];     // set-up
};

// One owned pair: [0] the even cell, [1] the odd one.
template <typename CT>
struct TailPair {
    CT d[2], inv[2], xp[2], xm[2], yp[2], ym[2], zp[2], zm[2];
    int id[2];        // padded indices (a second cell outside the level: d < 0)
    int pid;          // padded index of the parent on the next level, -1: none
    int ch;           // padded index of the first cell's first child on the level above
    bool valid, ok1, first_odd;   // pair exists; its second cell is inside the level; colour of its first cell
};

// Record loads of a pair (undefined where the pair does not exist).
template <int D, typename CT>
struct TailRecV {
    typename TailRec<CT>::Q v[TailRec<CT>::NV];
    int4 ix;
};
template <int D, typename CT>
__device__ __forceinline__ void tail_issue_rec(TailRecV<D, CT>& R, const void* rec, int rq, int p, int np) {
    using Q = typename TailRec<CT>::Q;
    constexpr int NV = TailRec<CT>::NV;
    const Q* base = static_cast<const Q*>(rec) + rq + p;
    const int st = tail_rec_stride(np);
    R.ix = int4{0, -1, 0, 0};
#pragma unroll
    for (int q = 0; q < NV; q++) R.v[q] = Q{};
    if (p < np) {
#pragma unroll
        for (int q = 0; q < (D == 3 ? NV : NV * 3 / 4); q++) R.v[q] = gload(base + q * st);   // 2D: no z couplings
        R.ix = __builtin_bit_cast(int4, gload(base + NV * st));
    }
}
template <int D, typename CT>
__device__ __forceinline__ void tail_pair_from_rec(TailPair<CT>& P, const TailRecV<D, CT>& R, int p, int np) {
    constexpr int PER = TailRec<CT>::PER;
    auto val = [&](int e) -> CT {
        const auto& q = R.v[e / PER];
        if constexpr (sizeof(CT) == 4) return (e & 3) == 0 ? q.x : ((e & 3) == 1 ? q.y : ((e & 3) == 2 ? q.z : q.w));
        else return (e & 1) ? q.y : q.x;
    };
#pragma unroll
    for (int c = 0; c < 2; c++) {
        P.d[c] = val(c); P.inv[c] = val(2 + c);
        P.xp[c] = val(4 + c); P.xm[c] = val(6 + c); P.yp[c] = val(8 + c); P.ym[c] = val(10 + c);
        P.zp[c] = val(12 + c); P.zm[c] = val(14 + c);
    }
    P.valid = p < np;
    P.first_odd = (R.ix.w & 1) != 0;
    P.ok1 = (R.ix.w & 2) != 0;
    P.id[0] = R.ix.x + (P.first_odd ? 1 : 0);
    P.id[1] = R.ix.x + (P.first_odd ? 0 : 1);
    P.pid = R.ix.y;
    P.ch = R.ix.z;
}

// Set-up: the records of the tail (TAIL_MAXP workgroups for the first level, one
// for every other).
template <int D, typename CT, typename C4>
__global__ __launch_bounds__(TAIL_THREADS) void k_tail_records(TailArgs<C4> A, CT* __restrict__ rec) {
    const int slot = blockIdx.x;
    const int l = slot < TAIL_MAXP ? 0 : slot - TAIL_MAXP + 1;
    const int v = slot < TAIL_MAXP ? slot : 0;
    if (l >= A.nl) return;
    const int t = threadIdx.x, p = t + TAIL_THREADS * v;
    const Geo g = A.g[l];
    if (p >= A.np[l]) return;
    const int npx = (g.nx + 1) >> 1;
    const int i0 = 2 * (p % npx) + 1, j = (p / npx) % g.ny + 1, k = (D == 3) ? p / (npx * g.ny) + 1 : 0;
    const int id0 = (int)gidx(g, i0, j, k), par0 = (i0 + j + k) & 1;
    const bool ok1 = i0 + 1 <= g.nx;
    constexpr int PER = TailRec<CT>::PER, NV = TailRec<CT>::NV;
    CT f[NV * PER];
#pragma unroll
    for (int c = 0; c < 2; c++) {   // cell of colour c
        const int q = c ^ par0;
        Sten<CT> s;
        s.d = CT(-1); s.xp = s.xm = s.yp = s.ym = s.zp = s.zm = CT(0);
        if (q == 0 || ok1) s = sten_lc<D, CT>(A.coef[l], g, id0 + q);
        f[c] = s.d;
        f[2 + c] = s.d >= CT(1e-30) ? recip(s.d) : CT(0);
        f[4 + c] = s.xp; f[6 + c] = s.xm; f[8 + c] = s.yp; f[10 + c] = s.ym;
        f[12 + c] = D == 3 ? s.zp : CT(0); f[14 + c] = D == 3 ? s.zm : CT(0);
    }
    const long at = A.rq[l] + p, st = tail_rec_stride(A.np[l]);
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
        for (int e = 0; e < PER; e++) rec[(at + q * st) * PER + e] = f[q * PER + e];
    int4 ix;
    ix.x = id0;
    ix.y = -1;
    if (l + 1 < A.nl) {
        const Geo cg = A.g[l + 1];
        const int ic = (i0 + 1) >> 1, jc = (j + 1) >> 1, kc = (D == 3) ? (k + 1) >> 1 : 0;
        if (ic <= cg.nx && jc <= cg.ny && (D != 3 || kc <= cg.nz)) ix.y = (int)gidx(cg, ic, jc, kc);
    }
    ix.z = l > 0 ? (int)gidx(A.g[l - 1], 2 * i0 - 1, 2 * j - 1, (D == 3) ? 2 * k - 1 : 0) : 0;
    ix.w = par0 | (ok1 ? 2 : 0);
    reinterpret_cast<int4*>(rec)[at + NV * st] = ix;
}

// One RBGS colour on the owned pairs of one level.
template <int D, int C, typename CT, int NP>
__device__ __forceinline__ void tail_smooth(const TailPair<CT> (&P)[NP], CT* X, const CT* Bv, int sx, int sy) {
#pragma unroll
    for (int v = 0; v < NP; v++) {
        const TailPair<CT>& p = P[v];
        if (p.inv[C] == CT(0)) continue;           // absent, solid or isolated
        const int id = p.id[C];
        CT nb = p.xp[C] * X[id + 1] + p.xm[C] * X[id - 1] + p.yp[C] * X[id + sx] + p.ym[C] * X[id - sx];
        if (D == 3) nb = nb + p.zp[C] * X[id + sy] + p.zm[C] * X[id - sy];
        X[id] = rdiv(Bv[id] + nb, p.d[C], p.inv[C]);
    }
}

// b - A x on the owned fluid cells (0 elsewhere), formed as k_restrict forms it.
template <int D, typename CT, int NP>
__device__ __forceinline__ void tail_residual(const TailPair<CT> (&P)[NP], const CT* X, const CT* Bv, CT* Rs, int sx, int sy) {
#pragma unroll
    for (int v = 0; v < NP; v++) {
        const TailPair<CT>& p = P[v];
        if (!p.valid) continue;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            if (!p.ok1 && (p.first_odd ? c == 0 : c == 1)) continue;   // the second cell, outside the level
            const int id = p.id[c];
            CT res = CT(0);
            if (p.d[c] >= CT(0)) {
                double Ax = (double)p.d[c] * (double)X[id] - (double)p.xp[c] * (double)X[id + 1]
                          - (double)p.xm[c] * (double)X[id - 1] - (double)p.yp[c] * (double)X[id + sx]
                          - (double)p.ym[c] * (double)X[id - sx];
                if (D == 3) Ax = Ax - (double)p.zp[c] * (double)X[id + sy] - (double)p.zm[c] * (double)X[id - sy];
                res = (CT)((double)Bv[id] - Ax);
            }
            Rs[id] = res;
        }
    }
}

// x_f += 2 x_c on the owned fluid cells whose parent lies in the coarse level.
template <typename CT, int NP>
__device__ __forceinline__ void tail_prolong(const TailPair<CT> (&P)[NP], CT* X, const CT* XC) {
#pragma unroll
    for (int v = 0; v < NP; v++) {
        const TailPair<CT>& p = P[v];
        if (p.pid < 0) continue;
        const CT xc = XC[p.pid];
#pragma unroll
        for (int c = 0; c < 2; c++)
            if (p.valid && p.d[c] >= CT(0)) X[p.id[c]] = X[p.id[c]] + CT(2) * xc;
    }
}

// b / d on the odd cells (the first pass of a level, whose x is 0)
template <typename CT>
__device__ __forceinline__ void tail_first(const TailPair<CT>& p, CT* X, CT b) {
    if (p.inv[1] != CT(0)) X[p.id[1]] = rdiv(b + CT(0), p.d[1], p.inv[1]);
}

// b of the owned pair = sum of the children's residuals (all its cells in the
// level), then the first pass (unless no pass is asked for on the coarsest).
template <int D, typename CT>
__device__ __forceinline__ void tail_restrict(const TailPair<CT>& p, const CT* Rs, CT* B, CT* X, int fsx, int fsy, bool first) {
    if (!p.valid) return;
    CT b[2];   // first and second cell
#pragma unroll
    for (int q = 0; q < 2; q++) {
        double sum = 0;
        if (q == 0 || p.ok1) {
            const CT* R = Rs + p.ch + 2 * q;
            for (int di = 0; di < 2; di++)
                for (int dj = 0; dj < 2; dj++)
                    for (int dk = 0; dk < (D == 3 ? 2 : 1); dk++) sum += (double)R[di + dj * fsx + dk * fsy];
        }
        b[q] = (CT)sum;
    }
    const int id0 = p.first_odd ? p.id[1] : p.id[0];
    B[id0] = b[0];
    if (p.ok1) B[id0 + 1] = b[1];
    if (first) tail_first(p, X, p.first_odd ? b[0] : b[1]);
}

template <int D, typename S, typename C4, int NLMAX>
__device__ __forceinline__ void d_tail(const TailArgs<C4>& Ag, bool test) {
    static_assert(NLMAX >= 2 && NLMAX <= TAIL_MAXL, "tail depth");
    using CT = typename CTOf<S>::type;
    __shared__ __align__(16) CT lds[TAIL_LDS_BYTES / sizeof(CT)];
    __shared__ TailArgs<C4> A;      // geometry and offsets (one vector load per dword)
    __shared__ double s_rr[FIN_THREADS / WAVE];
    const int tid = threadIdx.x;
    const int nl = Ag.nl;   // 1 <= nl <= NLMAX (checked on the host); 1: the coarsest level only
    const S* __restrict__ b_first = static_cast<const S*>(Ag.b);
    S* __restrict__ x_first = static_cast<S*>(Ag.x);
    int np[NLMAX];
#pragma unroll
    for (int l = 0; l < NLMAX; l++) np[l] = Ag.np[l];   // 0 past nl

    // every global load of the kernel's start first: the records of the
    // owned pairs (the first tail level has up to 2 pairs per thread, the
    // others 1) and b of the first level (at most TAIL_BMAX per thread,
    // checked on the host)
    TailRecV<D, CT> R0[TAIL_MAXP], R1, R2, R3, R4;
#pragma unroll
    for (int v = 0; v < TAIL_MAXP; v++) tail_issue_rec<D, CT>(R0[v], Ag.rec, Ag.rq[0], tid + TAIL_THREADS * v, np[0]);
    // FP64 (twice the registers): the levels below the second are loaded after
    // the first is done, and the first again for its way up (16 x 8 x 8: 13.9 ->
    // 12.2 us; a fourth 2D level still spilled 92 registers, 28 us)
    constexpr bool LATE = sizeof(CT) == 8;
    tail_issue_rec<D, CT>(R1, Ag.rec, Ag.rq[1], tid, np[1]);
    auto issue_rest = [&]() {
        if constexpr (NLMAX > 2) tail_issue_rec<D, CT>(R2, Ag.rec, Ag.rq[2], tid, np[2]);
        if constexpr (NLMAX > 3) tail_issue_rec<D, CT>(R3, Ag.rec, Ag.rq[3], tid, np[3]);
        if constexpr (NLMAX > 4) tail_issue_rec<D, CT>(R4, Ag.rec, Ag.rq[4], tid, np[4]);
    };
    if constexpr (!LATE) issue_rest();
    constexpr int BMAX = sizeof(CT) == 8 ? TAIL_LDS_BYTES / 24 / TAIL_THREADS : TAIL_BMAX;
    S bt[BMAX];
    const int N0 = Ag.N0;
#pragma unroll
    for (int u = 0; u < BMAX; u++) {
        const int e = tid + TAIL_THREADS * u;
        if (e < N0) bt[u] = gload(b_first + e);
    }
    // a vector load (the index lives in a VGPR), so that the flag is waited
    // for where it is tested, not at once by a scalar branch
    int skipped = 0;
    if (Ag.skip) {
        int z = 0;
        asm volatile("" : "+v"(z));
        skipped = gload(Ag.skip + z);
    }
    double rs = 0.0;
    FinState fs{};
    if (test) {
        fs = fin_state(Ag.ctrl);
        if (tid < FIN_THREADS)   // the finish kernel's order
            for (int e = tid; e < Ag.nrr; e += FIN_THREADS) rs += gload(Ag.rr + e);
    }
    {
        constexpr int NW = (int)(sizeof(TailArgs<C4>) / 4);
        static_assert(NW <= TAIL_THREADS && sizeof(TailArgs<C4>) % 4 == 0, "tail arguments");
        if (tid < NW) reinterpret_cast<uint32_t*>(&A)[tid] = reinterpret_cast<const uint32_t*>(&Ag)[tid];
    }
    // x = 0 on every level (ghosts included) while the loads are in flight;
    // the other arrays lie behind or between and are written before they are read
    for (int e = tid; e < Ag.ro; e += TAIL_THREADS) lds[e] = CT(0);
    __syncthreads();
    {
        CT* B0 = lds + A.bo[0];
#pragma unroll
        for (int u = 0; u < BMAX; u++) {
            const int e = tid + TAIL_THREADS * u;
            if (e < N0) B0[e] = (CT)bt[u];
        }
    }
    if (test && tid < FIN_THREADS) {
        rs = wave_sum(rs);
        if ((tid & (WAVE - 1)) == 0) s_rr[tid / WAVE] = rs;
    }
    TailPair<CT> P0[TAIL_MAXP], P1[1], P2[1], P3[1], P4[1];
    auto pairs_first = [&]() {
#pragma unroll
        for (int v = 0; v < TAIL_MAXP; v++) tail_pair_from_rec<D, CT>(P0[v], R0[v], tid + TAIL_THREADS * v, np[0]);
    };
    pairs_first();
    tail_pair_from_rec<D, CT>(P1[0], R1, tid, np[1]);
    auto pairs_rest = [&]() {
        if constexpr (NLMAX > 2) tail_pair_from_rec<D, CT>(P2[0], R2, tid, np[2]);
        if constexpr (NLMAX > 3) tail_pair_from_rec<D, CT>(P3[0], R3, tid, np[3]);
        if constexpr (NLMAX > 4) tail_pair_from_rec<D, CT>(P4[0], R4, tid, np[4]);
    };
    if constexpr (!LATE) pairs_rest();
    __syncthreads();
    if (test) {   // every thread takes the same decision from the same values, thread 0 stores it
        double tot = s_rr[0];
        for (int w = 1; w < FIN_THREADS / WAVE; w++) tot += s_rr[w];
        skipped |= fin_update_scalars(tid == 0 ? Ag.ctrl : nullptr, fs, tot);
    }
    if (skipped) return;   // uniform: every thread read the same flag

    // per-level offsets and strides, uniform
    auto u32 = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    struct Lev { CT *X, *B; int sx, sy; };
    auto level = [&](int l) { return Lev{lds + u32(A.xo[l]), lds + u32(A.bo[l]), u32((int)A.g[l].sx), u32((int)A.g[l].sy)}; };
    CT* Rs = lds + u32(A.ro);
    const bool w0 = u32(tid >> 6) == 0;
    // levels of at most 64 pairs (every one after the first such level): all
    // pairs belong to wave 0, whose LDS accesses complete in program order;
    // the fences keep the compiler from moving them across passes
    auto wave = [&](int l) { return np[l] <= WAVE; };
    auto sync = [&](bool w) {
        if (w) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            __syncthreads();
        }
    };
    // the first pass of level l is done; leaves the first pass of level l + 1 done
    auto level_down = [&](auto& P, auto& PC, int l) {
        const bool w = wave(l);
        if (w && !w0) return;
        const Lev L = level(l), C = level(l + 1);
        sync(w);
        tail_smooth<D, 0>(P, L.X, L.B, L.sx, L.sy);
        sync(w);
        tail_residual<D>(P, L.X, L.B, Rs, L.sx, L.sy);
        sync(w);
        tail_restrict<D>(PC[0], Rs, C.B, C.X, L.sx, L.sy, l + 2 < nl || A.npass > 0);
    };
    auto level_coarsest = [&](auto& P, int l) {   // odd, even, odd, ... (forward/reverse pairs collapsed)
        const bool w = wave(l);
        if (w && !w0) return;
        const Lev L = level(l);
        const int npass = u32(A.npass);
        int s = 1;                                 // the first pass is done
        for (; s + 1 < npass; s += 2) {
            sync(w);
            tail_smooth<D, 0>(P, L.X, L.B, L.sx, L.sy);
            sync(w);
            tail_smooth<D, 1>(P, L.X, L.B, L.sx, L.sy);
        }
        if (s < npass) { sync(w); tail_smooth<D, 0>(P, L.X, L.B, L.sx, L.sy); }
    };
    auto level_up = [&](auto& P, int l) {
        const bool w = wave(l);
        if (w && !w0) return;
        const Lev L = level(l);
        sync(w);
        tail_prolong(P, L.X, lds + u32(A.xo[l + 1]));
        sync(w);
        tail_smooth<D, 0>(P, L.X, L.B, L.sx, L.sy);
        sync(w);
        tail_smooth<D, 1>(P, L.X, L.B, L.sx, L.sy);
    };
    if (nl > 1 || A.npass > 0) {
        const CT* B0 = lds + u32(A.bo[0]);
#pragma unroll
        for (int v = 0; v < TAIL_MAXP; v++)
            if (P0[v].valid) tail_first(P0[v], lds + u32(A.xo[0]), B0[P0[v].id[1]]);
    }
    // down
    if (nl > 1) level_down(P0, P1, 0);
    if constexpr (LATE) { issue_rest(); pairs_rest(); }
    if constexpr (NLMAX > 2) { if (nl > 2) level_down(P1, P2, 1); }
    if constexpr (NLMAX > 3) { if (nl > 3) level_down(P2, P3, 2); }
    if constexpr (NLMAX > 4) { if (nl > 4) level_down(P3, P4, 3); }
    // coarsest
    if (nl == 1) level_coarsest(P0, 0);
    if (nl == 2) level_coarsest(P1, 1);
    if constexpr (NLMAX > 2) { if (nl == 3) level_coarsest(P2, 2); }
    if constexpr (NLMAX > 3) { if (nl == 4) level_coarsest(P3, 3); }
    if constexpr (NLMAX > 4) { if (nl == 5) level_coarsest(P4, 4); }
    // up
    if constexpr (NLMAX > 4) { if (nl > 4) level_up(P3, 3); }
    if constexpr (NLMAX > 3) { if (nl > 3) level_up(P2, 2); }
    if constexpr (LATE) {
        if (nl > 1) {
#pragma unroll
            for (int v = 0; v < TAIL_MAXP; v++) tail_issue_rec<D, CT>(R0[v], Ag.rec, Ag.rq[0], tid + TAIL_THREADS * v, np[0]);
            pairs_first();
        }
    }
    if constexpr (NLMAX > 2) { if (nl > 2) level_up(P1, 1); }
    if (nl > 1) level_up(P0, 0);
    // a thread stores its own cells (its last pass wrote the odd ones, the
    // pass before the even ones); ghosts of x are 0 from its allocation
    const CT* X0 = lds + u32(A.xo[0]);
#pragma unroll
    for (int v = 0; v < TAIL_MAXP; v++) {
        if (!P0[v].valid) continue;
        const int id0 = P0[v].first_odd ? P0[v].id[1] : P0[v].id[0];
        gstore(x_first + id0, (S)X0[id0]);
        if (P0[v].ok1) gstore(x_first + id0 + 1, (S)X0[id0 + 1]);
    }
}

template <int D, typename S, typename C4, int NLMAX>
__global__ __launch_bounds__(TAIL_THREADS) void k_tail(TailArgs<C4> A) {
    d_tail<D, S, C4, NLMAX>(A, A.rr != nullptr);
}

}  // namespace uaamg
