// kernels_gmg.hpp -- the GMG and AMG preconditioners of the reference's
// other factory keys ("pcg" / "pcg_gmg": GMGPreconditioner; "pcg_amg":
// AMGPreconditioner), 2D.
//
// Both build the same 2x2 hierarchy with a rediscretised 5-point operator
// per level (h doubles per level), a coarse cell solid when at least two of
// its four children are, and V(2,2) cycles with 10 x (forward + reverse)
// sweeps on the coarsest level (gmg_preconditioner.cpp:13-194,
// amg_preconditioner.cpp:13-209).  The smoother updates one colour in place:
//   x += (b - diag x + lap) / d_eff,  lap = (xL + xR)/dx^2 + (xB + xT)/dy^2
// with a wall or solid neighbour taking the cell's own value and d_eff the
// diagonal without those faces.  Restriction is the mean of the fluid
// children's residuals; AMG writes the residual as b - (diag x - lap) and
// every coarse cell, GMG as (b - diag x) + lap and only fluid coarse cells.
// Prolongation adds the parent's x to the fluid children.  The arithmetic
// and its order are the reference's, so the FP64 form matches it bit for bit.
#pragma once
#include "kernels_tile.hpp"

namespace uaamg {

// per-level constants of the rediscretised operator (host computes them as
// the reference does: GMG diag = 2 (1/dx^2 + 1/dy^2), AMG 2/dx^2 + 2/dy^2)
template <typename CT>
struct GmgC {
    CT idx2, idy2, diag;
};

// ---------------------------------------------------------------- fused passes
//
// One kernel per level on the way down (both forward sweeps, the residual
// and the restriction), one on the way up (the prolongation and both reverse
// sweeps), and one workgroup for the small levels.
//
// These levels are latency-bound like the UAAMG ones (kernels_tile.hpp), with
// four colour passes a launch, so the pass is kept short.  A workgroup owns
// GT_X x GT_Y cells and a halo of GT_H; a thread owns two neighbouring cells
// of a row, one of each colour, with x, b, the face flags and 1 / eff_d in its
// registers.  A pass reads its side neighbour from the lane beside it (DPP),
// the two vertical ones from LDS, and writes one value: each colour pass
// spoils one ring of the region, going down the first none (x = 0).  A wave
// holds rows of one parity, so which cell of the pair a pass updates is a
// scalar branch.  1 / eff_d comes from a table of the 16 neighbour patterns.
// At 500 x 390 FP64 a down launch takes 5.8 us and an up launch 5.4 (tile
// passes over LDS arrays of x, b, flags and 1 / eff_d with eight cells a
// thread: 14.0 and 13.6), the small levels 38.9 (49.8 without per-cell
// flags and 1 / eff_d); 88 us per PCG iteration instead of 187.

constexpr int GT_H = 4, GT_RX = 64, GT_RY = 32, GT_X = GT_RX - 2 * GT_H, GT_Y = GT_RY - 2 * GT_H, GT_THREADS = 1024;
constexpr int GMG_TAIL_THREADS = 1024, GMG_TAIL_MAXL = 8;
constexpr int GMG_TAIL_PAIRS = 4;                        // pairs a thread owns on a level, at most
constexpr int GMG_TAIL_LDS = 150 * 1024;                 // bytes of x, b, 1 / eff_d and flags of the tail levels

// Face flags of a cell: bit 0 fluid, bits 1-4 the neighbour at +x, -x, +y, -y
// takes part (the neighbour byte's bits); a wall or solid neighbour gives the
// cell's own value and drops its face from the diagonal.
constexpr uint8_t GF_FLUID = NB_FLUID, GF_XP = NB_XP, GF_XM = NB_XM, GF_YP = NB_YP, GF_YM = NB_YM;

// 1 / eff_d of a neighbour pattern, eff_d formed as the smoother forms it
// (gmg_preconditioner.cpp:41-81, amg_preconditioner.cpp:13-50)
template <typename CT>
__device__ __forceinline__ CT gmg_inv_d(uint8_t f, const GmgC<CT>& c) {
    CT eff_d = c.diag;
    if (!(f & GF_XM)) eff_d -= c.idx2;
    if (!(f & GF_XP)) eff_d -= c.idx2;
    if (!(f & GF_YM)) eff_d -= c.idy2;
    if (!(f & GF_YP)) eff_d -= c.idy2;
    return (eff_d < CT(1e-15)) ? CT(0) : CT(1) / eff_d;
}
// one cell's update, the reference smoother's arithmetic in its order
template <typename CT>
__device__ __forceinline__ CT gmg_update(CT xc, CT xL, CT xR, CT xB, CT xT, CT b, uint8_t f, CT d, const GmgC<CT>& c) {
    xL = (f & GF_XM) ? xL : xc;
    xR = (f & GF_XP) ? xR : xc;
    xB = (f & GF_YM) ? xB : xc;
    xT = (f & GF_YP) ? xT : xc;
    const CT lap = (xL + xR) * c.idx2 + (xB + xT) * c.idy2;
    return xc + d * (b - c.diag * xc + lap);
}
// the residual of one cell as the restriction forms it (GMG (b - diag x) +
// lap, gmg_preconditioner.cpp:121-142; AMG b - (diag x - lap),
// amg_preconditioner.cpp:91-111)
template <bool AMG, typename CT>
__device__ __forceinline__ CT gmg_resid(CT xc, CT xL, CT xR, CT xB, CT xT, CT b, uint8_t f, const GmgC<CT>& c) {
    xL = (f & GF_XM) ? xL : xc;
    xR = (f & GF_XP) ? xR : xc;
    xB = (f & GF_YM) ? xB : xc;
    xT = (f & GF_YP) ? xT : xc;
    if constexpr (AMG) {
        const CT Ax = c.diag * xc - (xL + xR) * c.idx2 - (xB + xT) * c.idy2;
        return b - Ax;
    } else {
        const CT lap = (xL + xR) * c.idx2 + (xB + xT) * c.idy2;
        return b - c.diag * xc + lap;
    }
}
// b of a coarse cell from its children's residuals (0 on solid ones), in the
// order (0,0), (0,1), (1,0), (1,1)
template <bool AMG, typename CT, typename VC>
__device__ __forceinline__ void gmg_put_coarse(CT r00, CT r01, CT r10, CT r11, int cnt, VC* bc, bool solid) {
    const CT sum = CT(0) + r00 + r01 + r10 + r11;
    if constexpr (AMG) *bc = (VC)((cnt > 0) ? sum / (CT)cnt : CT(0));
    else if (!solid && cnt > 0) *bc = (VC)(sum / (CT)cnt);
}

template <typename CT>
struct GmgLDS {
    CT x[2][GT_THREADS];      // [left / right cell][row * 32 + pair]
    uint8_t fl[GT_THREADS];   // bit 0 / 1: the left / right cell is fluid
    CT tab[16];               // 1 / eff_d per neighbour pattern
};
template <typename CT>
struct GmgPair {
    int hx, rj, e, gi, gj;
    bool in0, in1, own, lo;   // lo (uniform over the wave): the left cell is odd
    long id;
    uint8_t f0, f1;
    CT x0, x1, b0, b1, d0, d1;
    __device__ __forceinline__ void init(const Geo& g, int bx, int by) {
        const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
        hx = lane & 31;
        rj = 4 * (w >> 1) + (w & 1) + 2 * (lane >> 5);   // rows r and r + 2
        lo = (w & 1) != 0;                               // gi and gj of row 0 are odd
        e = rj * 32 + hx;
        gi = bx * GT_X + 1 - GT_H + 2 * hx;
        gj = by * GT_Y + 1 - GT_H + rj;
        const bool row = gj >= 1 && gj <= g.ny;
        in0 = row && gi >= 1 && gi <= g.nx;
        in1 = in0 && gi + 1 <= g.nx;                     // gi is odd
        own = hx >= GT_H / 2 && hx < 32 - GT_H / 2 && rj >= GT_H && rj < GT_RY - GT_H;
        id = gi + gj * g.sx;
        x0 = x1 = b0 = b1 = CT(0);
    }
    // flags from the solid mask (which the ghost layer need not be part of)
    __device__ __forceinline__ void flags(const uint8_t* __restrict__ S, const Geo& g) {
        uint8_t m0 = 1, m1 = 1, u0 = 1, u1 = 1, v0 = 1, v1 = 1, side = 1;
        if (in0) {
            t2_pair(S + id, m0, m1);
            if (gj > 1) t2_pair(S + id - g.sx, u0, u1);
            if (gj < g.ny) t2_pair(S + id + g.sx, v0, v1);
            if (hx == 0 && gi > 1) side = S[id - 1];
            if (hx == 31 && gi + 1 < g.nx) side = S[id + 2];
        }
        if (!in1) m1 = 1;
        // the cells beside the pair: solid or outside there reads as 1
        const int pk = (m0 ? 1 : 0) | (m1 ? 2 : 0);
        int l = __builtin_amdgcn_update_dpp(3, pk, 0x138, 0xF, 0xF, false) >> 1;   // lane - 1's right cell
        int r = __builtin_amdgcn_update_dpp(3, pk, 0x130, 0xF, 0xF, false) & 1;    // lane + 1's left cell
        if (hx == 0) l = side ? 1 : 0;
        if (hx == 31) r = side ? 1 : 0;
        f0 = f1 = 0;
        if (!m0) f0 = (uint8_t)(GF_FLUID | (m1 ? 0 : GF_XP) | (l ? 0 : GF_XM) | (v0 ? 0 : GF_YP) | (u0 ? 0 : GF_YM));
        if (!m1) f1 = (uint8_t)(GF_FLUID | (r ? 0 : GF_XP) | (m0 ? 0 : GF_XM) | (v1 ? 0 : GF_YP) | (u1 ? 0 : GF_YM));
    }
    // one colour pass on the cells at least `ring` inside the region
    template <bool RIGHT>
    __device__ __forceinline__ void cell(GmgLDS<CT>& L, int ring, const GmgC<CT>& c) {
        const CT side = RIGHT ? lane_from_right(x0) : lane_from_left(x1);   // all lanes take part
        const int col = 2 * hx + (RIGHT ? 1 : 0);
        const uint8_t f = RIGHT ? f1 : f0;
        if (!(f & GF_FLUID) || col < ring || col >= GT_RX - ring || rj < ring || rj >= GT_RY - ring) return;
        const CT* X = L.x[RIGHT];
        const CT xB = rj > 0 ? X[e - 32] : CT(0), xT = rj < GT_RY - 1 ? X[e + 32] : CT(0);
        CT& x = RIGHT ? x1 : x0;
        x = gmg_update<CT>(x, RIGHT ? x0 : side, RIGHT ? side : x1, xB, xT, RIGHT ? b1 : b0, f, RIGHT ? d1 : d0, c);
        L.x[RIGHT][e] = x;
    }
    __device__ __forceinline__ void pass(GmgLDS<CT>& L, bool odd, int ring, const GmgC<CT>& c) {
        if (odd == lo) cell<false>(L, ring, c);
        else cell<true>(L, ring, c);
        __syncthreads();
    }
};

// Down: x = 0, smooth twice (odd, even colours), restrict the residual; x
// of the tile (to xd) and the coarse b written.
template <bool AMG, typename VX, typename VC>
__global__ __launch_bounds__(GT_THREADS) void k_gmg_down(VX* __restrict__ xd, const VX* __restrict__ b,
                                                         const uint8_t* __restrict__ S, Geo g,
                                                         GmgC<typename CTOf<VX>::type> c, VC* __restrict__ bc,
                                                         const uint8_t* __restrict__ SC, Geo cg, const int* skip) {
    using CT = typename CTOf<VX>::type;
    __shared__ GmgLDS<CT> L;
    const int stop = skip ? *skip : 0;
    const int t = tile_of_block(), nbx = (g.nx + GT_X - 1) / GT_X;
    if (t >= nbx * ((g.ny + GT_Y - 1) / GT_Y)) return;
    GmgPair<CT> p;
    p.init(g, t % nbx, t / nbx);
    if (p.in0) {
        VX v0, v1;
        t2_pair(b + p.id, v0, v1);
        p.b0 = (CT)v0;
        p.b1 = (CT)v1;
    }
    const int ic = (p.gi + 1) >> 1, jc = (p.gj + 1) >> 1;
    const bool put = p.own && !(p.rj & 1) && ic <= cg.nx && jc <= cg.ny;
    const long cid = ic + jc * cg.sx;
    const bool csolid = put && SC[cid];
    p.flags(S, g);
    if (stop) return;
    if (threadIdx.x < 16) L.tab[threadIdx.x] = gmg_inv_d<CT>((uint8_t)(threadIdx.x << 1), c);
    L.x[0][p.e] = L.x[1][p.e] = CT(0);
    L.fl[p.e] = (uint8_t)((p.f0 & GF_FLUID) | ((p.f1 & GF_FLUID) << 1));
    __syncthreads();
    p.d0 = L.tab[p.f0 >> 1];
    p.d1 = L.tab[p.f1 >> 1];
    for (int q = 0; q < 4; q++) p.pass(L, !(q & 1), q, c);
    if (p.own && p.in0) t2_put(xd + p.id, (VX)p.x0, (VX)p.x1, p.in1);
    // residuals of the tile; the odd rows' go through LDS
    const CT xl = lane_from_left(p.x1), xr = lane_from_right(p.x0);
    CT r0 = CT(0), r1 = CT(0);
    if (p.own) {
        if (p.f0 & GF_FLUID) r0 = gmg_resid<AMG, CT>(p.x0, xl, p.x1, L.x[0][p.e - 32], L.x[0][p.e + 32], p.b0, p.f0, c);
        if (p.f1 & GF_FLUID) r1 = gmg_resid<AMG, CT>(p.x1, p.x0, xr, L.x[1][p.e - 32], L.x[1][p.e + 32], p.b1, p.f1, c);
    }
    __syncthreads();
    if (p.rj & 1) { L.x[0][p.e] = r0; L.x[1][p.e] = r1; }
    __syncthreads();
    if (put) {
        const int cnt = __popc((unsigned)L.fl[p.e]) + __popc((unsigned)L.fl[p.e + 32]);
        gmg_put_coarse<AMG, CT, VC>(r0, L.x[0][p.e + 32], r1, L.x[1][p.e + 32], cnt, bc + cid, csolid);
    }
}

// Up: x = xd + the parent's x on fluid cells (GMG: fluid parents only), smooth
// twice in reverse (even, odd colours); x of the tile written to xo (another
// buffer: other workgroups still read xd on their halo).
template <bool AMG, typename VX, typename VC>
__global__ __launch_bounds__(GT_THREADS) void k_gmg_up(const VX* __restrict__ xd, VX* __restrict__ xo, const VX* __restrict__ b,
                                                       const uint8_t* __restrict__ S, Geo g,
                                                       GmgC<typename CTOf<VX>::type> c, const VC* __restrict__ xcoarse,
                                                       const uint8_t* __restrict__ SC, Geo cg, const int* skip) {
    using CT = typename CTOf<VX>::type;
    __shared__ GmgLDS<CT> L;
    const int stop = skip ? *skip : 0;
    const int t = tile_of_block(), nbx = (g.nx + GT_X - 1) / GT_X;
    if (t >= nbx * ((g.ny + GT_Y - 1) / GT_Y)) return;
    GmgPair<CT> p;
    p.init(g, t % nbx, t / nbx);
    const int ic = (p.gi + 1) >> 1, jc = (p.gj + 1) >> 1;
    bool hp = p.in0 && ic <= cg.nx && jc <= cg.ny;   // a parent
    CT xp = CT(0);
    uint8_t pm = 1;
    if (p.in0) {
        VX v0, v1;
        t2_pair(b + p.id, v0, v1);
        p.b0 = (CT)v0;
        p.b1 = (CT)v1;
        t2_pair(xd + p.id, v0, v1);
        p.x0 = (CT)v0;
        p.x1 = p.in1 ? (CT)v1 : CT(0);
    }
    if (hp) { xp = (CT)xcoarse[ic + jc * cg.sx]; pm = SC[ic + jc * cg.sx]; }
    p.flags(S, g);
    if (stop) return;
    hp = hp && (AMG || !pm);
    if (hp && (p.f0 & GF_FLUID)) p.x0 = (CT)(VX)(p.x0 + xp);   // prolongateAdd (gmg :144-156, amg :113-123)
    if (hp && (p.f1 & GF_FLUID)) p.x1 = (CT)(VX)(p.x1 + xp);
    if (threadIdx.x < 16) L.tab[threadIdx.x] = gmg_inv_d<CT>((uint8_t)(threadIdx.x << 1), c);
    L.x[0][p.e] = p.x0;
    L.x[1][p.e] = p.x1;
    __syncthreads();
    p.d0 = L.tab[p.f0 >> 1];
    p.d1 = L.tab[p.f1 >> 1];
    for (int q = 0; q < 4; q++) p.pass(L, q & 1, q + 1, c);
    if (p.own && p.in0) t2_put(xo + p.id, (VX)p.x0, (VX)p.x1, p.in1);
}

// The small levels in one workgroup: x, b, 1 / eff_d and face flags of every
// tail level in LDS, the V-cycle below the first tail level run pass by pass
// with workgroup barriers (gmg_vcycle from the first tail level down).  A
// thread owns the same pairs of cells throughout.
struct GmgTailArgs {
    int nl;                              // levels in the tail; the last is the coarsest
    Geo g[GMG_TAIL_MAXL];
    GmgC<double> c[GMG_TAIL_MAXL];
    const uint8_t* mask[GMG_TAIL_MAXL];  // padded solid masks (device)
    int off[GMG_TAIL_MAXL];              // LDS element offset of each level's arrays
    int total;                           // padded cells of all tail levels
    int csweeps;                         // coarsest (forward + reverse) pairs
    // the convergence test of this iteration, as in k_tail
    const double* rr;
    int nrr;
    Ctrl* ctrl;
};

// End of a tail phase: the whole workgroup, or (levels with at most 64
// pairs, run by wave 0 alone) wave order only -- the LDS accesses of one wave
// complete in program order; the fences keep the compiler from moving them
// across phases.
__device__ __forceinline__ void gmg_tail_sync(bool wave) {
    if (wave) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// A level's geometry and arrays, and a thread's pairs on it: e[v] is the left
// cell of pair v (0: none), left_odd its colour, v < NP.
template <typename CT, int NP>
struct GmgTailLevel {
    GmgC<CT> c;
    CT *X, *B, *D;
    uint8_t* F;
    int sx, e[NP];
    bool lo[NP], in1[NP];
    __device__ __forceinline__ void init(const GmgTailArgs& A, int l, CT* Xa, CT* Ba, CT* Da, uint8_t* Fa) {
        const Geo g = A.g[l];
        c = GmgC<CT>{(CT)A.c[l].idx2, (CT)A.c[l].idy2, (CT)A.c[l].diag};
        X = Xa + A.off[l]; B = Ba + A.off[l]; D = Da + A.off[l]; F = Fa + A.off[l];
        sx = (int)g.sx;
        const int npx = (g.nx + 1) >> 1, np = npx * g.ny;
#pragma unroll
        for (int v = 0; v < NP; v++) {
            const int p = (int)threadIdx.x + v * GMG_TAIL_THREADS;
            const int i = 2 * (p % npx) + 1, j = p / npx + 1;
            e[v] = p < np ? i + j * sx : 0;
            lo[v] = ((i + j) & 1) != 0;
            in1[v] = i + 1 <= g.nx;
        }
    }
    __device__ __forceinline__ void colour(bool odd) const {
#pragma unroll
        for (int v = 0; v < NP; v++) {
            const bool right = lo[v] != odd;
            if (e[v] == 0 || (right && !in1[v])) continue;
            const int k = e[v] + (right ? 1 : 0);
            const uint8_t f = F[k];
            const CT xc = X[k], xl = X[k - 1], xr = X[k + 1], xb = X[k - sx], xt = X[k + sx], b = B[k], d = D[k];
            if (f & GF_FLUID) X[k] = gmg_update<CT>(xc, xl, xr, xb, xt, b, f, d, c);
        }
    }
    __device__ __forceinline__ void smooth(bool reverse, int sweeps, bool wave) const {
        for (int s = 0; s < sweeps; s++) {
            colour(!reverse);
            gmg_tail_sync(wave);
            colour(reverse);
            gmg_tail_sync(wave);
        }
    }
    template <bool AMG>
    __device__ __forceinline__ CT resid(int k) const {
        const uint8_t f = F[k];
        return (f & GF_FLUID) ? gmg_resid<AMG, CT>(X[k], X[k - 1], X[k + 1], X[k - sx], X[k + sx], B[k], f, c) : CT(0);
    }
};

// the coarsest level's passes with at most 64 pairs, in wave 0: everything
// but the neighbours' x stays in registers
template <typename CT>
__device__ __forceinline__ void gmg_tail_coarsest(const GmgTailLevel<CT, 1>& L, int csweeps) {
    const int k0 = L.e[0];
    const bool on = k0 != 0, lo = L.lo[0];
    uint8_t fo = 0, fe = 0;       // flags, b, 1 / eff_d, x of the odd and the even cell
    CT bo = CT(0), be = CT(0), dO = CT(0), de = CT(0), xo = CT(0), xe = CT(0);
    const int ko = lo ? k0 : k0 + 1, ke = lo ? k0 + 1 : k0;
    if (on && (lo || L.in1[0])) { fo = L.F[ko]; bo = L.B[ko]; dO = L.D[ko]; xo = L.X[ko]; }
    if (on && (!lo || L.in1[0])) { fe = L.F[ke]; be = L.B[ke]; de = L.D[ke]; xe = L.X[ke]; }
    auto one = [&](int k, uint8_t f, CT b, CT d, CT& x, CT y) {
        if (f & GF_FLUID) {
            const bool right = k != k0;
            const CT s = L.X[right ? k + 1 : k - 1], xb = L.X[k - L.sx], xt = L.X[k + L.sx];
            x = gmg_update<CT>(x, right ? y : s, right ? s : y, xb, xt, b, f, d, L.c);
            L.X[k] = x;
        }
        gmg_tail_sync(true);
    };
    for (int s = 0; s < csweeps; s++) {   // forward (odd, even), reverse (even, odd)
        one(ko, fo, bo, dO, xo, xe);
        one(ke, fe, be, de, xe, xo);
        one(ke, fe, be, de, xe, xo);
        one(ko, fo, bo, dO, xo, xe);
    }
}

template <bool AMG, typename VF, typename CT = typename CTOf<VF>::type>
__global__ __launch_bounds__(GMG_TAIL_THREADS) void k_gmg_tail(GmgTailArgs A_, VF* __restrict__ x0,
                                                               const VF* __restrict__ b0, const int* skip) {
    __shared__ __align__(16) unsigned char lds[GMG_TAIL_LDS];
    __shared__ GmgTailArgs A;   // copied in one round trip, as in d_tail
    __shared__ int s_stop;
    const int tid = (int)threadIdx.x;
    constexpr int NW = (int)(sizeof(GmgTailArgs) / 4);
    static_assert(NW <= GMG_TAIL_THREADS && sizeof(GmgTailArgs) % 4 == 0, "tail arguments");
    if (tid < NW) reinterpret_cast<uint32_t*>(&A)[tid] = reinterpret_cast<const uint32_t*>(&A_)[tid];
    const int skipped = skip ? *skip : 0;
    __syncthreads();
    CT* Xa = reinterpret_cast<CT*>(lds);
    CT* Ba = Xa + A.total;
    CT* Da = Ba + A.total;
    uint8_t* Fa = reinterpret_cast<uint8_t*>(Da + A.total);
    double rs[1] = {0.0};
    FinState fs{};
    if (A.rr && tid == 0) fs = fin_state(A.ctrl);
    if (A.rr && tid < FIN_THREADS)   // the finish kernel's order
        for (int e = tid; e < A.nrr; e += FIN_THREADS) rs[0] += gload(A.rr + e);
    const int nl = A.nl;
    for (int l = 0; l < nl; l++) {
        const Geo g = A.g[l];
        const int off = A.off[l];
        for (int e = tid; e < (int)g.N; e += GMG_TAIL_THREADS) {
            const int gi = e % (int)g.sx, gj = e / (int)g.sx;
            const bool in = gi >= 1 && gi <= g.nx && gj >= 1 && gj <= g.ny;
            Fa[off + e] = in && !A.mask[l][e] ? GF_FLUID : 0;
            Xa[off + e] = CT(0);
            Ba[off + e] = (l == 0 && in) ? (CT)b0[e] : CT(0);
        }
    }
    __syncthreads();
    if (A.rr) {
        block_sum<1>(rs);
        if (tid == 0) s_stop = fin_update_scalars(A.ctrl, fs, rs[0]);
        __syncthreads();
        if (s_stop) return;
    }
    if (skipped) return;
    // face flags (bit 0 of the neighbours is written by no one here) and 1 / eff_d
    for (int l = 0; l < nl; l++) {
        const Geo g = A.g[l];
        const int off = A.off[l], sx = (int)g.sx;
        const GmgC<CT> c{(CT)A.c[l].idx2, (CT)A.c[l].idy2, (CT)A.c[l].diag};
        for (int e = tid; e < (int)g.N; e += GMG_TAIL_THREADS) {
            uint8_t* F = Fa + off + e;
            if (!(*F & GF_FLUID)) continue;
            const uint8_t f = (uint8_t)(GF_FLUID | ((F[1] & GF_FLUID) ? GF_XP : 0) | ((F[-1] & GF_FLUID) ? GF_XM : 0) |
                                        ((F[sx] & GF_FLUID) ? GF_YP : 0) | ((F[-sx] & GF_FLUID) ? GF_YM : 0));
            *F = f;
            Da[off + e] = gmg_inv_d<CT>(f, c);
        }
    }
    __syncthreads();
    auto restrict_to = [&](const auto& L, int l, bool wave) {   // level l -> l + 1
        const int nt = wave ? 64 : GMG_TAIL_THREADS;
        const Geo cg = A.g[l + 1];
        for (int t = tid; t < cg.nx * cg.ny; t += nt) {
            const int ic = 1 + t % cg.nx, jc = 1 + t / cg.nx;
            const int k = 2 * ic - 1 + (2 * jc - 1) * L.sx, cid = A.off[l + 1] + ic + jc * (int)cg.sx;
            const int cnt = (L.F[k] & 1) + (L.F[k + 1] & 1) + (L.F[k + L.sx] & 1) + (L.F[k + L.sx + 1] & 1);
            gmg_put_coarse<AMG, CT, CT>(L.template resid<AMG>(k), L.template resid<AMG>(k + L.sx), L.template resid<AMG>(k + 1),
                                        L.template resid<AMG>(k + L.sx + 1), cnt, Ba + cid, !(Fa[cid] & GF_FLUID));
        }
        gmg_tail_sync(wave);
    };
    auto prolong_from = [&](const auto& L, int l, bool wave) {   // level l + 1 -> l
        const Geo cg = A.g[l + 1];
        const CT* XC = Xa + A.off[l + 1];
        const uint8_t* FC = Fa + A.off[l + 1];
        constexpr int NP = (int)(sizeof(L.e) / sizeof(int));
#pragma unroll
        for (int v = 0; v < NP; v++) {
            const int k = L.e[v];
            if (k == 0) continue;
            const int ic = (k % L.sx + 1) >> 1, jc = (k / L.sx + 1) >> 1;   // both cells of the pair share the parent
            if (ic > cg.nx || jc > cg.ny) continue;
            const int cid = ic + jc * (int)cg.sx;
            if (!AMG && !(FC[cid] & GF_FLUID)) continue;
            if (L.F[k] & GF_FLUID) L.X[k] = L.X[k] + XC[cid];
            if (L.in1[v] && (L.F[k + 1] & GF_FLUID)) L.X[k + 1] = L.X[k + 1] + XC[cid];
        }
        gmg_tail_sync(wave);
    };
    auto pairs = [&](int l) { return A.g[l].ny * ((A.g[l].nx + 1) >> 1); };
    // levels [0, lw) on the workgroup, [lw, nl) on wave 0 (lw = nl: a coarsest
    // level of more than 64 pairs, on the workgroup)
    int lw = nl;
    for (int l = nl - 1; l >= 0 && pairs(l) <= 64; l--) lw = l;
    const int top = lw < nl - 1 ? lw : nl - 1;
    GmgTailLevel<CT, GMG_TAIL_PAIRS> L;
    for (int l = 0; l < top; l++) {
        L.init(A, l, Xa, Ba, Da, Fa);
        L.smooth(false, 2, false);
        restrict_to(L, l, false);
    }
    if (lw < nl) {
        if (tid < 64) {
            GmgTailLevel<CT, 1> W;
            for (int l = top; l < nl - 1; l++) {
                W.init(A, l, Xa, Ba, Da, Fa);
                W.smooth(false, 2, true);
                restrict_to(W, l, true);
            }
            W.init(A, nl - 1, Xa, Ba, Da, Fa);
            gmg_tail_coarsest<CT>(W, A.csweeps);
            for (int l = nl - 2; l >= top; l--) {
                W.init(A, l, Xa, Ba, Da, Fa);
                prolong_from(W, l, true);
                W.smooth(true, 2, true);
            }
        }
        __syncthreads();
    } else {
        L.init(A, nl - 1, Xa, Ba, Da, Fa);
        for (int s = 0; s < A.csweeps; s++) { L.smooth(false, 1, false); L.smooth(true, 1, false); }
    }
    for (int l = top - 1; l >= 0; l--) {
        L.init(A, l, Xa, Ba, Da, Fa);
        prolong_from(L, l, false);
        L.smooth(true, 2, false);
    }
    const Geo g0 = A.g[0];
    for (int e = tid; e < (int)g0.N; e += GMG_TAIL_THREADS) {
        const int gi = e % (int)g0.sx, gj = e / (int)g0.sx;
        if (gi >= 1 && gi <= g0.nx && gj >= 1 && gj <= g0.ny) x0[e] = (VF)Xa[e];
    }
}

}  // namespace uaamg
