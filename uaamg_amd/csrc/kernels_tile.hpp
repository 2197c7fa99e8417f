// kernels_tile.hpp -- the 2D V(1,1) level kernels, one launch down and one up
// per level with a workgroup per tile, and the 2D CG passes around them.
//
// Same arithmetic and order per cell as the per-pass kernels (and so the
// reference's smooth / restrictResidual / prolongateAdd,
// uaamg_preconditioner.cpp:107-175).  2D levels are latency-bound: a 512 x 256
// FP64 level is 1 MB, so what counts is the chain load - sweep - sweep -
// store, not the bytes.  A workgroup loads its tile and two cells of halo at
// once and a thread owns two neighbouring cells of a row (one of each colour,
// both children of one coarse cell):
//   * values and stencils stay in its registers;
//   * the left and right neighbours come from the lanes beside it by DPP, the
//     ones above and below through LDS, the restriction's second row from
//     lane + 32 (a wave holds two rows of 32 pairs);
//   * two barriers per launch, one for each colour.
// The march kernels that ran here before went through the level row by row
// with four barriers a row.  At 1024 x 512 FP64: down 11.9 -> 6.1 us, level-0 up
// 13.2 -> 9.3, the four coarse levels above the tail 5.5 -> 4.0 each way (a
// launch with nothing in it takes 2.2); with the fused CG passes 17 launches
// and 108 us per iteration became 11 and 80.
#pragma once
#include "kernels_cg.hpp"
#include "kernels_march.hpp"
#include "kernels_rows.hpp"

namespace uaamg {

// Region of 64 x 16 cells, tile of 60 x 12 (68 % of the threads own a cell
// that counts): eight waves, so a 1024 x 512 level is 774 workgroups and the
// chip holds all of them at once.
constexpr int T2_X = 60, T2_Y = 12, T2_THREADS = 512;
__host__ __device__ constexpr int t2_nx(const Geo& g) { return (g.nx + T2_X - 1) / T2_X; }
__host__ __device__ constexpr int t2_tiles(const Geo& g) { return t2_nx(g) * ((g.ny + T2_Y - 1) / T2_Y); }

// Tile of block b of a single-grid launch: XCD-first, as row_tile_of_block
// (the tiles of one XCD are neighbours and share their halo in its L2).
inline unsigned tile_blocks(long tiles) { return 8u * (unsigned)((tiles + 7) / 8); }
__device__ __forceinline__ int tile_of_block() { return (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)); }

// Two neighbouring values in one load; the first lies in the level, the second
// in the level or its ghost layer.
template <typename V>
__device__ __forceinline__ void t2_pair(const V* __restrict__ p, V& a, V& b) {
    typedef V V2 __attribute__((ext_vector_type(2), aligned(sizeof(V))));
    const V2 v = *(const V2*)p;
    a = v[0];
    b = v[1];
}
template <typename V>
__device__ __forceinline__ void t2_put(V* __restrict__ p, V a, V b, bool second) {
    typedef V V2 __attribute__((ext_vector_type(2), aligned(sizeof(V))));
    if (second) *(V2*)p = V2{a, b};
    else *p = a;
}

template <typename CT>
struct T2St { CT xp, xm, yp, ym, d; };   // one cell; d < 0: not fluid

template <typename CT>
struct T2LDS {
    CT x[2][T2_THREADS];     // [left / right cell of the pair][pair]
    CT cy[2][T2_THREADS];    // Lc: +y couplings
};

// The position of a thread's pair; the left cell is (gi, gj), gi odd.
struct T2Pos {
    int gi, gj, e, hx, rj;
    bool in0, in1, own, r0, r1, left_odd;   // r0 / r1: the cells have all neighbours in the region
    long id;
    __device__ __forceinline__ void init(const Geo& g, int bx, int by) {
        e = (int)threadIdx.x;
        hx = e & 31;
        rj = e >> 5;
        gi = bx * T2_X - 1 + 2 * hx;
        gj = by * T2_Y - 1 + rj;
        const bool row = gj >= 1 && gj <= g.ny;
        in0 = row && gi >= 1 && gi <= g.nx;
        in1 = row && gi + 1 >= 1 && gi + 1 <= g.nx;
        const bool rr = rj >= 1 && rj <= 14;
        r0 = rr && hx >= 1;
        r1 = rr && hx <= 30;
        own = hx >= 1 && hx <= 30 && rj >= 2 && rj <= 13;
        left_odd = ((gi + gj) & 1) != 0;
        id = gi + gj * g.sx;
    }
};

// The stencils of the pair: level 0 from the neighbour bytes, levels >= 1 from
// the records; their -x coupling is the left cell's +x, their -y coupling
// (the row above's +y) is read from LDS after the first barrier.
template <bool L0, typename CT, typename C4>
__device__ __forceinline__ void t2_load_stencil(const FusedArgs<2, L0, CT, C4>& A, const T2Pos& t, T2St<CT>& s0, T2St<CT>& s1) {
    if constexpr (L0) {
        uint8_t n0 = 0, n1 = 0;
        if (t.in0) t2_pair(A.nbr + t.id, n0, n1);
        if (!t.in1) n1 = 0;
        const auto a = msten0<2, CT>(n0, A.c, A.g, t.gi, t.gj, 0);
        const auto b = msten0<2, CT>(n1, A.c, A.g, t.gi + 1, t.gj, 0);
        s0 = T2St<CT>{a.ap, a.am, a.mp, a.mm, a.d};
        s1 = T2St<CT>{b.ap, b.am, b.mp, b.mm, b.d};
    } else {
        s0 = T2St<CT>{CT(0), CT(0), CT(0), CT(0), CT(-1)};
        s1 = s0;
        if (t.in0) { const C4 r = A.rec[t.id]; s0.xp = (CT)r.x; s0.yp = (CT)r.y; s0.d = (CT)r.w; }
        if (t.in1) { const C4 r = A.rec[t.id + 1]; s1.xp = (CT)r.x; s1.yp = (CT)r.y; s1.d = (CT)r.w; }
        s0.xm = lane_from_left(s1.xp);
        s1.xm = s0.xp;
    }
}

// one colour of the pair: its cell's update where the colour and the ring allow it
template <bool L0, typename CT>
__device__ __forceinline__ void t2_sweep(T2LDS<CT>& S, const T2Pos& t, bool right, bool on, CT& x0, CT& x1, CT b0, CT b1,
                                         const T2St<CT>& s0, const T2St<CT>& s1) {
    const CT xl = lane_from_left(x1), xr = lane_from_right(x0);   // all lanes: DPP reads the neighbours' registers
    const CT d = right ? s1.d : s0.d;
    if (on && d >= CT(1e-30)) {
        const CT* X = S.x[right];
        const CT up = X[t.e + 32], dn = X[t.e - 32];
        const CT ap = right ? s1.xp : s0.xp, am = right ? s1.xm : s0.xm;
        const CT mp = right ? s1.yp : s0.yp, mm = right ? s1.ym : s0.ym;
        const CT nb = ap * (right ? xr : x1) + am * (right ? x0 : xl) + mp * up + mm * dn;
        const CT v = mdiv<CT>((right ? b1 : b0) + nb, d);
        if (right) x1 = v;
        else x0 = v;
    }
}
template <typename CT>
__device__ __forceinline__ void t2_lds_ym(const T2LDS<CT>& S, const T2Pos& t, T2St<CT>& s0, T2St<CT>& s1) {
    const int e = t.rj >= 1 ? t.e - 32 : t.e;
    s0.ym = S.cy[0][e];
    s1.ym = S.cy[1][e];
}

// Down: forward sweep from x = 0, residual, restriction (b of the next level).
template <bool L0, typename VB, typename C4, typename VC>
__device__ __forceinline__ void d_t2_down(const VB* __restrict__ b, const FusedArgs<2, L0, typename CTOf<VB>::type, C4>& A,
                                          VC* __restrict__ bc, const Geo& cg, int bx, int by) {
    using CT = typename CTOf<VB>::type;
    __shared__ T2LDS<CT> S;
    T2Pos t;
    t.init(A.g, bx, by);
    T2St<CT> s0, s1;
    CT b0 = CT(0), b1 = CT(0);
    if (t.in0) {   // gi is odd: in1 alone cannot be
        VB v0, v1;
        t2_pair(b + t.id, v0, v1);
        b0 = (CT)v0;
        b1 = t.in1 ? (CT)v1 : CT(0);
    }
    t2_load_stencil<L0, CT, C4>(A, t, s0, s1);
    // odd cells: x = b / d
    CT x0 = (t.left_odd && s0.d >= CT(1e-30)) ? mdiv<CT>(b0 + CT(0), s0.d) : CT(0);
    CT x1 = (!t.left_odd && s1.d >= CT(1e-30)) ? mdiv<CT>(b1 + CT(0), s1.d) : CT(0);
    S.x[0][t.e] = x0;
    S.x[1][t.e] = x1;
    if constexpr (!L0) { S.cy[0][t.e] = s0.yp; S.cy[1][t.e] = s1.yp; }
    __syncthreads();
    if constexpr (!L0) t2_lds_ym(S, t, s0, s1);
    // even cells.  A vertical neighbour has the other colour, so every value
    // read here was written before the barrier, and every one written here is
    // read after the next.
    t2_sweep<L0, CT>(S, t, t.left_odd, t.left_odd ? t.r1 : t.r0, x0, x1, b0, b1, s0, s1);
    S.x[t.left_odd][t.e] = t.left_odd ? x1 : x0;
    __syncthreads();
    // residual b - A x of the tile's fluid cells
    const CT xl = lane_from_left(x1), xr = lane_from_right(x0);
    CT q0 = CT(0), q1 = CT(0);
    if (t.own) {
        if (s0.d >= CT(0)) {
            CT Ax = s0.d * x0 - s0.xp * x1 - s0.xm * xl;
            Ax = Ax - s0.yp * S.x[0][t.e + 32] - s0.ym * S.x[0][t.e - 32];
            q0 = b0 - Ax;
        }
        if (s1.d >= CT(0)) {
            CT Ax = s1.d * x1 - s1.xp * xr - s1.xm * x0;
            Ax = Ax - s1.yp * S.x[1][t.e + 32] - s1.ym * S.x[1][t.e - 32];
            q1 = b1 - Ax;
        }
    }
    // the coarse cell's children: this pair and the one below it, lane + 32
    const CT q2 = __shfl_down(q0, 32, 64), q3 = __shfl_down(q1, 32, 64);
    if (t.own && !(t.rj & 1)) {
        const int ic = (t.gi + 1) >> 1, jc = (t.gj + 1) >> 1;
        if (ic <= cg.nx && jc <= cg.ny) bc[ic + jc * cg.sx] = (VC)(q0 + q2 + q1 + q3);
    }
}

// Up: x' = x0 + 2 x_coarse, reverse sweep.  Level 0 (of batch members; single
// grids: d_t2_up0): with the z sums (sum z, sum r z, sum r over fluid cells) of
// the tile in partials[q np].
template <bool L0, typename VB, typename C4, typename VCX>
__device__ __forceinline__ void d_t2_up(const VB* __restrict__ b, const FusedArgs<2, L0, typename CTOf<VB>::type, C4>& A,
                                        const VCX* __restrict__ xc, const Geo& cg, VB* __restrict__ xout, int bx, int by,
                                        double* partials = nullptr, int np = 0) {
    using CT = typename CTOf<VB>::type;
    __shared__ T2LDS<CT> S;
    T2Pos t;
    t.init(A.g, bx, by);
    T2St<CT> s0, s1;
    CT b0 = CT(0), b1 = CT(0), c = CT(0);
    if (t.in0) {   // gi is odd: in1 alone cannot be
        VB v0, v1;
        t2_pair(b + t.id, v0, v1);
        b0 = (CT)v0;
        b1 = t.in1 ? (CT)v1 : CT(0);
    }
    {
        const int ic = (t.gi + 1) >> 1, jc = (t.gj + 1) >> 1;
        if (t.in0 && ic <= cg.nx && jc <= cg.ny) c = (CT)xc[ic + jc * cg.sx];
    }
    t2_load_stencil<L0, CT, C4>(A, t, s0, s1);
    CT x0 = (t.left_odd && s0.d >= CT(1e-30)) ? mdiv<CT>(b0 + CT(0), s0.d) : CT(0);
    CT x1 = (!t.left_odd && s1.d >= CT(1e-30)) ? mdiv<CT>(b1 + CT(0), s1.d) : CT(0);
    if (s0.d >= CT(0)) x0 = x0 + CT(2) * c;
    if (s1.d >= CT(0)) x1 = x1 + CT(2) * c;
    S.x[0][t.e] = x0;
    S.x[1][t.e] = x1;
    if constexpr (!L0) { S.cy[0][t.e] = s0.yp; S.cy[1][t.e] = s1.yp; }
    __syncthreads();
    if constexpr (!L0) t2_lds_ym(S, t, s0, s1);
    t2_sweep<L0, CT>(S, t, t.left_odd, t.left_odd ? t.r1 : t.r0, x0, x1, b0, b1, s0, s1);   // even cells
    S.x[t.left_odd][t.e] = t.left_odd ? x1 : x0;
    __syncthreads();
    t2_sweep<L0, CT>(S, t, !t.left_odd, t.own, x0, x1, b0, b1, s0, s1);                     // odd cells
    if (t.own && t.in0) t2_put(xout + t.id, (VB)x0, (VB)x1, t.in1);
    if constexpr (L0) {
        double red[3] = {0.0, 0.0, 0.0};
        if (t.own && s0.d >= CT(0)) { const double z = (double)(VB)x0, r = (double)b0; red[0] = z; red[1] = r * z; red[2] = r; }
        if (t.own && s1.d >= CT(0)) { const double z = (double)(VB)x1, r = (double)b1; red[0] += z; red[1] += r * z; red[2] += r; }
        block_sum<3>(red);
        if (threadIdx.x == 0)
            for (int q = 0; q < 3; q++) partials[(long)q * np] = red[q];
    }
}

template <bool L0, typename VB, typename C4, typename VC>
__global__ __launch_bounds__(T2_THREADS) void k_t2_down(const VB* __restrict__ b, FusedArgs<2, L0, typename CTOf<VB>::type, C4> A,
                                                        VC* __restrict__ bc, Geo cg, const int* skip) {
    if (skip && *skip) return;
    const int t = tile_of_block();
    if (t >= t2_tiles(A.g)) return;
    d_t2_down<L0, VB, C4, VC>(b, A, bc, cg, t % t2_nx(A.g), t / t2_nx(A.g));
}
template <typename VB, typename C4>
__global__ __launch_bounds__(T2_THREADS) void k_t2_up(const VB* __restrict__ b, FusedArgs<2, false, typename CTOf<VB>::type, C4> A,
                                                      const VB* __restrict__ xc, Geo cg, VB* __restrict__ xout, const int* skip) {
    if (skip && *skip) return;
    const int t = tile_of_block();
    if (t < t2_tiles(A.g)) d_t2_up<false, VB, C4, VB>(b, A, xc, cg, xout, t % t2_nx(A.g), t / t2_nx(A.g));
}

// ---------------------------------------------------------------- level 0, up
// The same with the z sums (sum z, sum r z, sum r over fluid cells).  Their
// order decides the last digits of every CG scalar, so it is the march
// kernel's: a workgroup owns 252 columns and KC rows (that kernel's chunk),
// each column is added from the top down and the columns as block_store adds
// them.  512 threads, 128 pairs a row, row rj + 4 u for u < U (KC + 4 <= 4 U);
// all neighbours come from LDS here (a row spans two waves).  1/d comes from a
// table of the 16 neighbour patterns (rdiv, kernels_vcycle.hpp).  Chunks of more than 12 rows
// (grids of about 2.5 million cells and more) stay on the march kernel, whose
// halo rows then cost little.
constexpr int T2U_RX = 256, T2U_HX = 128, T2U_MAXU = 4;

template <int U, typename VB, typename VCX>
__device__ __forceinline__ void d_t2_up0(const VB* __restrict__ b, const uint8_t* __restrict__ nbr, const Geo& g,
                                         const Consts<typename CTOf<VB>::type>& cc, const VCX* __restrict__ xc, const Geo& cg,
                                         VB* __restrict__ xout, int KC, int bx, int bz, double* partials, int np) {
    using CT = typename CTOf<VB>::type;
    __shared__ CT X[2][4 * U * T2U_HX];     // [left / right cell][row * 128 + pair]
    __shared__ CT Rv[2][4 * U * T2U_HX];    // r, for the column sums
    __shared__ CT tab[2][16];               // d and 1/d per neighbour pattern, without walls
    const int hx = (int)threadIdx.x & (T2U_HX - 1);
    const int rg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 7);   // uniform: so are the row tests and the colours
    const int gi = bx * (T2U_RX - 4) - 1 + 2 * hx, m0 = bz * KC + 1, last = min(m0 + KC - 1, g.ny), nr = last - m0 + 5;
    CT x0[U], x1[U], b0[U], b1[U], d0[U], d1[U], i0[U], i1[U], cx[U];
    uint8_t n0[U], n1[U];
    const int ic = (gi + 1) >> 1;
    const bool c0 = gi >= 1 && gi <= g.nx, c1 = gi + 1 >= 1 && gi + 1 <= g.nx;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int gj = m0 - 2 + rg + 4 * u, jc = (gj + 1) >> 1;
        const bool row = gj >= 1 && gj <= g.ny && rg + 4 * u < nr;
        const long id = gi + gj * g.sx;
        b0[u] = b1[u] = cx[u] = CT(0);
        n0[u] = n1[u] = 0;
        if (row && c0) {   // gi is odd: c1 alone cannot be
            VB v0, v1;
            t2_pair(b + id, v0, v1);
            b0[u] = (CT)v0;
            b1[u] = (CT)v1;
            t2_pair(nbr + id, n0[u], n1[u]);
            if (!c1) { b1[u] = CT(0); n1[u] = 0; }
            if (ic <= cg.nx && jc <= cg.ny) cx[u] = (CT)xc[ic + jc * cg.sx];
        }
    }
    if (threadIdx.x < 16) {
        Consts<CT> k = cc;
        k.any_dirichlet = 0;
        const CT d = msten0<2, CT>((uint8_t)(NB_FLUID | (threadIdx.x << 1)), k, g, 2, 2, 0).d;
        tab[0][threadIdx.x] = d;
        tab[1][threadIdx.x] = d >= CT(1e-30) ? recip(d) : CT(0);
    }
    __syncthreads();
    // d, and 1/d (0 on cells that no sweep updates: solid or isolated)
#pragma unroll
    for (int u = 0; u < U; u++) {
        d0[u] = tab[0][(n0[u] >> 1) & 15]; i0[u] = tab[1][(n0[u] >> 1) & 15];
        d1[u] = tab[0][(n1[u] >> 1) & 15]; i1[u] = tab[1][(n1[u] >> 1) & 15];
        if (cc.any_dirichlet) {
            const int gj = m0 - 2 + rg + 4 * u;
            d0[u] = msten0<2, CT>(n0[u], cc, g, gi, gj, 0).d;
            d1[u] = msten0<2, CT>(n1[u], cc, g, gi + 1, gj, 0).d;
            i0[u] = d0[u] >= CT(1e-30) ? recip(d0[u]) : CT(0);
            i1[u] = d1[u] >= CT(1e-30) ? recip(d1[u]) : CT(0);
        }
        if (!(n0[u] & NB_FLUID)) i0[u] = CT(0);
        if (!(n1[u] & NB_FLUID)) i1[u] = CT(0);
    }
    // odd rows start with an odd left cell (the halo's two rows and 4 u do not matter)
    const bool lo = ((m0 + rg) & 1) == 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int e = (rg + 4 * u) * T2U_HX + hx;
        x0[u] = x1[u] = CT(0);
        if (lo) { if (i0[u] != CT(0)) x0[u] = rdiv(b0[u], d0[u], i0[u]); }
        else { if (i1[u] != CT(0)) x1[u] = rdiv(b1[u], d1[u], i1[u]); }
        if (n0[u] & NB_FLUID) x0[u] = x0[u] + CT(2) * cx[u]; else b0[u] = CT(0);
        if (n1[u] & NB_FLUID) x1[u] = x1[u] + CT(2) * cx[u]; else b1[u] = CT(0);
        X[0][e] = x0[u];
        X[1][e] = x1[u];
        Rv[0][e] = b0[u];
        Rv[1][e] = b1[u];
    }
    __syncthreads();
    // one colour of the rows, its cells left or right of the pairs; ring:
    // rows and columns inside the region by that much
    auto sweep = [&](auto right_, int ring) {
        constexpr bool right = decltype(right_)::value;
        if (right ? 2 * hx + 1 > T2U_RX - 1 - ring || 2 * hx + 1 < ring : 2 * hx < ring || 2 * hx > T2U_RX - 1 - ring) return;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int rj = rg + 4 * u, e = rj * T2U_HX + hx;
            if (rj < ring || rj >= nr - ring) continue;
            const uint8_t n = right ? n1[u] : n0[u];
            const CT side = right ? X[0][e + 1] : X[1][e - 1];
            const CT ap = (n & NB_XP) ? cc.idx2 : CT(0), am = (n & NB_XM) ? cc.idx2 : CT(0);
            const CT mp = (n & NB_YP) ? cc.idy2 : CT(0), mm = (n & NB_YM) ? cc.idy2 : CT(0);
            const CT nb = ap * (right ? side : x1[u]) + am * (right ? x0[u] : side) + mp * X[right][e + T2U_HX] + mm * X[right][e - T2U_HX];
            const CT inv = right ? i1[u] : i0[u];
            CT& x = right ? x1[u] : x0[u];
            if (inv != CT(0)) x = rdiv((right ? b1[u] : b0[u]) + nb, right ? d1[u] : d0[u], inv);
            X[right][e] = x;
        }
    };
    if (lo) sweep(std::true_type{}, 1);     // even cells
    else sweep(std::false_type{}, 1);
    __syncthreads();
    if (lo) sweep(std::false_type{}, 2);    // odd cells
    else sweep(std::true_type{}, 2);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int rj = rg + 4 * u, gj = m0 - 2 + rj;
        if (rj < 2 || rj >= nr - 2 || hx < 1 || hx > T2U_HX - 2) continue;
        const long id = gi + gj * g.sx;
        if (c0) t2_put(xout + id, (VB)x0[u], (VB)x1[u], c1);
    }
    // thread t < 256 adds column t of the region (its cells outside the level
    // and the fluid hold 0)
    double red[3] = {0.0, 0.0, 0.0};
    const int t = (int)threadIdx.x;
    if (t >= 2 && t < T2U_RX - 2) {
        for (int rj = 2; rj < nr - 2; rj++) {
            const int e = rj * T2U_HX + (t >> 1);
            const double zz = (double)(VB)X[t & 1][e], rr = (double)Rv[t & 1][e];
            red[0] += zz; red[1] += rr * zz; red[2] += rr;
        }
    }
    block_sum<3>(red);
    if (t == 0)
        for (int q = 0; q < 3; q++) partials[(long)q * np] = red[q];
}
template <int U, typename VB, typename VCX>
__global__ __launch_bounds__(512) void k_t2_up0(const VB* __restrict__ b, const uint8_t* __restrict__ nbr, Geo g,
                                                Consts<typename CTOf<VB>::type> c, const VCX* __restrict__ xc, Geo cg,
                                                VB* __restrict__ xout, int KC, int nbx, int np, const int* skip, double* partials) {
    if (skip && *skip) return;
    const int t = tile_of_block();   // nbx workgroups a row of them, np in all
    if (t >= np) return;
    d_t2_up0<U, VB, VCX>(b, nbr, g, c, xc, cg, xout, KC, t % nbx, t / nbx, partials + t, np);
}

// ---------------------------------------------------------------- CG passes
// Each of the three flat passes of an iteration takes over the finish of the
// launch before it: every workgroup (FIN_THREADS threads, as the finish
// kernels have) adds the partials in their order.  Cells, threads and sums
// are those of k_pupdate, k_matvec_dot and k_update, so every scalar is the
// same bit for bit.

// The loads of a thread's first vector and every scalar of the finish are
// issued before the partials are added: one memory round trip, not three
// (1024 x 512 FP64: operator 12.2 -> 9.9 us, update 7.9 -> 6.8 us).

// what the operator reads of z or p_old around the vector at c0 (3D: f, k:
// the planes below and above)
template <int D, typename T>
struct T2Nb { vec4<T> c, b, t, f, k; T l, r; };
template <int D, typename T>
__device__ __forceinline__ T2Nb<D, T> t2_nb(const T* __restrict__ v, long c0, const Geo& g) {
    T2Nb<D, T> o;
    o.c = *(const vec4<T>*)(v + c0);
    o.b = *(const vec4u<T>*)(v + c0 - g.sx);
    o.t = *(const vec4u<T>*)(v + c0 + g.sx);
    if constexpr (D == 3) {
        o.f = *(const vec4u<T>*)(v + c0 - g.sy);
        o.k = *(const vec4u<T>*)(v + c0 + g.sy);
    }
    o.l = v[c0 - 1];
    o.r = v[c0 + 4];
    return o;
}

// The finish of the z sums, p (written to the other p buffer: neighbours form
// theirs from p_old) and Ap with its p.Ap partials.  rsold and the first flag
// are read here and only written by the next launch.
template <int D, typename T, bool VAR>
__global__ __launch_bounds__(FIN_THREADS) void k_t2_pmv(const T* __restrict__ z, const T* __restrict__ pold, T* __restrict__ pnew,
                                                        T* __restrict__ Ap, const uint8_t* __restrict__ nbr, Geo g,
                                                        Consts<double> c, long N4, Ctrl* ctrl, const double* zp, int nz, double* pap,
                                                        VarLap L) {
    const int done = ctrl->done, project = ctrl->project, first = ctrl->first;
    const double count = ctrl->count, rsold = ctrl->rsold;
    const int fv_b = blockIdx.x, fv_n = gridDim.x;
    double tot[3] = {0.0, 0.0, 0.0};
    for (int x = threadIdx.x; x < nz; x += FIN_THREADS)
#pragma unroll
        for (int q = 0; q < 3; q++) tot[q] += zp[(long)q * nz + x];
    // FLAT_LOOP_XCD's range
    const long n = N4 / 4, len = (n + 7) / 8;
    const bool xcd = (fv_n & 7) == 0;
    const long beg = (xcd ? (fv_b & 7) * len + (long)(fv_b >> 3) * FIN_THREADS : (long)fv_b * FIN_THREADS) + threadIdx.x;
    const long end = xcd ? min(n, ((fv_b & 7) + 1) * len) : n;
    const long step = (long)(xcd ? (fv_n >> 3) : fv_n) * FIN_THREADS;
    const long first_v = min(beg, n - 1);          // a thread without a vector loads the last one
    uint32_t w = *(const uint32_t*)(nbr + 4 * first_v);
    // vectors of the first and the last plane, which hold no fluid cell, load
    // one whose neighbour planes lie in the array
    const long first_c = D == 3 ? min(max(4 * first_v, (g.sy + 3) / 4 * 4), (N4 - g.sy - 4) / 4 * 4) : 4 * first_v;
    T2Nb<D, T> zv = t2_nb<D, T>(z, first_c, g), pv = t2_nb<D, T>(pold, first_c, g);
    if (done) return;
    __shared__ double s_z[3];
    block_sum<3>(tot);
    if (threadIdx.x == 0) { s_z[0] = tot[0]; s_z[1] = tot[1]; s_z[2] = tot[2]; }
    __syncthreads();
    const double sz = s_z[0], srz = s_z[1], sr = s_z[2];
    const double mean = (project && count > 0) ? sz / count : 0.0;
    const double rz = srz - mean * sr;
    const double beta = first ? 0.0 : rz / rsold;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->sum_z = sz; ctrl->sum_rz = srz; ctrl->sum_r = sr;
        ctrl->mean_z = mean; ctrl->rz = rz; ctrl->beta = beta;
        if (!isfinite(rz)) { ctrl->done = 1; ctrl->status = ST_NONFINITE; }
    }
    // the whole solve stops: the launches after this one see done, and what a
    // workgroup that saw it half way wrote to p and Ap is read by none
    if (!isfinite(rz)) return;
    auto at = [&](T zz, T pp) { return (T)(((double)zz - mean) + beta * (double)pp); };
    double v[1] = {0.0};
    for (long k = beg; k < end; k += step) {
        const long c0 = 4 * k;
        if (k != beg) {
            w = *(const uint32_t*)(nbr + c0);
            if (w & 0x01010101u) { zv = t2_nb<D, T>(z, c0, g); pv = t2_nb<D, T>(pold, c0, g); }
        }
        vec4<T> out = (T)0;
        if (w & 0x01010101u) {
            vec4<T> po = (T)0;
            T pc[6];
            pc[0] = at(zv.l, pv.l);
            pc[5] = at(zv.r, pv.r);
#pragma unroll
            for (int q = 0; q < 4; q++) pc[q + 1] = at(zv.c[q], pv.c[q]);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint8_t nb = nbyte(w, q);
                if (!(nb & NB_FLUID)) continue;
                const double pm = (double)pc[q + 1], vl = (double)pc[q], vr = (double)pc[q + 2];
                const double vb = (double)at(zv.b[q], pv.b[q]), vt = (double)at(zv.t[q], pv.t[q]);
                double vf = 0.0, vk = 0.0;
                if constexpr (D == 3) { vf = (double)at(zv.f[q], pv.f[q]); vk = (double)at(zv.k[q], pv.k[q]); }
                double o;
                if constexpr (VAR) {
                    int i = 0, j = 0, kk = 0;
                    if (c.any_dirichlet) coords<2>(g, c0 + q, i, j, kk);
                    o = apply_A_var(i, j, c0 + q, nb, pm, vl, vr, vb, vt, g, c, L);
                } else {
                    o = apply_A<D>(c0 + q, nb, pm, vl, vr, vb, vt, vf, vk, g, c);
                }
                const T oq = (T)o;
                out[q] = oq;
                po[q] = pc[q + 1];
                v[0] += pm * (double)oq;
            }
            *(vec4<T>*)(pnew + c0) = po;   // nothing reads the p of the other cells
        }
        *(vec4<T>*)(Ap + c0) = out;
    }
    block_store<1>(v, pap);
}

// The operator's finish (alpha, breakdown), x += alpha p, r -= alpha Ap and
// the r.r partials.  Workgroup 0 stores the scalars, rsold for the next beta
// and a breakdown for the convergence test (Ctrl::status); no workgroup of this
// launch reads those.
template <typename T>
__global__ __launch_bounds__(FIN_THREADS) void k_t2_update(T* __restrict__ x, T* __restrict__ r, const T* __restrict__ p,
                                                           const T* __restrict__ Ap, const uint8_t* __restrict__ nbr, long N4,
                                                           int nvb, double* rr, const double* pap, int npap, Ctrl* ctrl) {
    const int done = ctrl->done;
    const double rz = ctrl->rz;
    double tot[1] = {0.0};
    for (int k = threadIdx.x; k < npap; k += FIN_THREADS) tot[0] += pap[k];
    // block vb of the flat pass runs on the XCD whose level-0 tiles hold its cells
    const int vb = tile_of_block();
    if (vb >= nvb) return;
    const long n = N4 / 4, beg = (long)vb * FIN_THREADS + threadIdx.x, step = (long)nvb * FIN_THREADS;
    const long c1 = 4 * min(beg, n - 1);
    uint32_t w = *(const uint32_t*)(nbr + c1);
    vec4<T> xv = *(const vec4<T>*)(x + c1), rv = *(const vec4<T>*)(r + c1), pv = *(const vec4<T>*)(p + c1), av = *(const vec4<T>*)(Ap + c1);
    if (done) return;
    __shared__ double s_pap;
    block_sum<1>(tot);
    if (threadIdx.x == 0) s_pap = tot[0];
    __syncthreads();
    const double pAp = s_pap;
    const bool ok = isfinite(pAp) && pAp >= 1e-15;   // pcg.cpp:100 breakdown test
    const double alpha = rz / pAp;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->pAp = pAp;
        if (!ok) ctrl->status = isfinite(pAp) ? ST_BREAKDOWN : ST_NONFINITE;
        ctrl->alpha = ctrl->xalpha = ok ? alpha : 0.0;
        ctrl->rsold = rz;
        ctrl->first = 0;
    }
    if (!ok) return;
    double v[1] = {0.0};
    for (long k = beg; k < n; k += step) {
        const long c = 4 * k;
        if (k != beg) {
            w = *(const uint32_t*)(nbr + c);
            if (w & 0x01010101u) {
                xv = *(const vec4<T>*)(x + c); rv = *(const vec4<T>*)(r + c);
                pv = *(const vec4<T>*)(p + c); av = *(const vec4<T>*)(Ap + c);
            }
        }
        if (!(w & 0x01010101u)) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (!(nbyte(w, q) & NB_FLUID)) continue;
            xv[q] = (T)((double)xv[q] + alpha * (double)pv[q]);
            const T rn = (T)((double)rv[q] - alpha * (double)av[q]);
            rv[q] = rn;
            v[0] += (double)rn * (double)rn;
        }
        *(vec4<T>*)(x + c) = xv;
        *(vec4<T>*)(r + c) = rv;
    }
    block_sum<1>(v);
    if (threadIdx.x == 0) rr[vb] = v[0];
}

}  // namespace uaamg
