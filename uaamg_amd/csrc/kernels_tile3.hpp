// kernels_tile3.hpp -- the 3D V(1,1) kernels of the record levels (1 and
// below), one launch down and one up per level with a workgroup per tile.
//
// Same arithmetic and order per cell as the per-pass kernels (and so the
// reference's smooth / restrictResidual / prolongateAdd,
// uaamg_preconditioner_3d.cpp:123-181).  Levels of up to 64^3 are bound by
// latency: the march kernels that ran here before took six plane steps with
// three barriers each for two planes of output.  A workgroup loads its tile
// and two cells of halo on every side at once; a thread owns the cells
// (i, i+1) x (k, k+1) of one row, so
//   * half of the vertical neighbours, both children of a coarse cell in x and
//     in z and all stencils are in its registers;
//   * the left and right neighbours come from the lanes beside it by DPP, the
//     other y and z neighbours through LDS, the restriction's second row from
//     lane + 32 (a wave holds two rows of 32 pairs);
//   * two barriers per launch, one for each colour.
// In FP32: 64^3 down 10.0 -> 6.5 us, up 10.5 -> 8.9 (beside the x update),
// 24 x 20 x 18 down 4.9 -> 4.0, up 4.0 (a launch with nothing in it takes 2.2).
#pragma once
#include "kernels_tile.hpp"

namespace uaamg {

// Region of 64 x 8 x 8 cells, tile of 4 x 4 rows: rows of at most 64 cells
// whole, longer ones in windows of 60 cells with two of halo on each side.
constexpr int T3_X = 64, T3_XW = 60, T3_T = 4, T3_THREADS = 1024, T3_SLOTS = 2048;
__host__ __device__ constexpr int t3_nx(const Geo& g) { return g.nx <= T3_X ? 1 : (g.nx + T3_XW - 1) / T3_XW; }
__host__ __device__ constexpr int t3_ny(const Geo& g) { return (g.ny + T3_T - 1) / T3_T; }
__host__ __device__ constexpr int t3_tiles(const Geo& g) { return t3_nx(g) * t3_ny(g) * ((g.nz + T3_T - 1) / T3_T); }

template <typename CT>
struct T3St { CT xp, xm, yp, ym, zp, zm, d; };   // one cell; d < 0: not fluid

template <typename CT>
struct T3LDS {
    CT x[2][T3_SLOTS];          // [left / right cell of the pair][plane * 256 + row * 32 + pair]
    CT cy[2][T3_SLOTS];         // +y couplings
    CT cz[2][T3_SLOTS / 2];     // +z couplings of a thread's upper plane
};

// A thread's four cells: pairs (gi, gi + 1), gi odd, on planes gk (odd) and gk + 1.
struct T3Pos {
    int gi, gj, gk, e, hx, rj, rk, ec;
    bool in0[2], in1[2], rr[2], own, own_wave, r0, r1, left_odd;   // left_odd: on plane gk; the other way round above
    long id[2];
    __device__ __forceinline__ void init(const Geo& g, int tile) {
        const int nwx = t3_nx(g), bx = tile % nwx, by = (tile / nwx) % t3_ny(g), bz = tile / (nwx * t3_ny(g));
        const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const bool whole = nwx == 1;
        hx = lane & 31;
        rj = 2 * (w & 3) + (lane >> 5);
        rk = 2 * (w >> 2);
        e = rk * 256 + rj * 32 + hx;
        ec = (rk >> 1) * 256 + rj * 32 + hx;
        gi = whole ? 1 + 2 * hx : bx * T3_XW - 1 + 2 * hx;
        gj = by * T3_T - 1 + rj;
        gk = bz * T3_T - 1 + rk;
        own_wave = ((w & 3) == 1 || (w & 3) == 2) && ((w >> 2) == 1 || (w >> 2) == 2);
        own = own_wave && (whole || (hx >= 1 && hx <= 30));
        r0 = whole || hx >= 1;      // the left / right cell has its x neighbours in the region
        r1 = whole || hx <= 30;
        left_odd = ((gj + gk) & 1) == 0;
        id[0] = gi + gj * g.sx + gk * g.sy;
        id[1] = id[0] + g.sy;
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const bool row = gj >= 1 && gj <= g.ny && gk + v >= 1 && gk + v <= g.nz;
            in0[v] = row && gi >= 1 && gi <= g.nx;
            in1[v] = row && gi + 1 <= g.nx && gi >= 1;
            rr[v] = rj >= 1 && rj <= 6 && rk + v >= 1 && rk + v <= 6;
        }
    }
};

template <typename CT> __device__ __forceinline__ CT t3_left(const T3Pos& t, CT v) { const CT l = lane_from_left(v); return t.hx == 0 ? CT(0) : l; }
template <typename CT> __device__ __forceinline__ CT t3_right(const T3Pos& t, CT v) { const CT r = lane_from_right(v); return t.hx == 31 ? CT(0) : r; }

// b and the records of the four cells; the -x coupling is the left cell's +x
template <typename VB, typename C4, typename CT>
__device__ __forceinline__ void t3_load(const VB* __restrict__ b, const C4* __restrict__ rec, const T3Pos& t, CT (&bv)[2][2], T3St<CT> (&s)[2][2]) {
#pragma unroll
    for (int v = 0; v < 2; v++) {
        bv[v][0] = bv[v][1] = CT(0);
        s[v][0] = T3St<CT>{CT(0), CT(0), CT(0), CT(0), CT(0), CT(0), CT(-1)};
        s[v][1] = s[v][0];
        if (t.in0[v]) {
            VB v0, v1;
            t2_pair(b + t.id[v], v0, v1);
            bv[v][0] = (CT)v0;
            bv[v][1] = t.in1[v] ? (CT)v1 : CT(0);
            const C4 r = rec[t.id[v]];
            s[v][0].xp = (CT)r.x; s[v][0].yp = (CT)r.y; s[v][0].zp = (CT)r.z; s[v][0].d = (CT)r.w;
        }
        if (t.in1[v]) {
            const C4 r = rec[t.id[v] + 1];
            s[v][1].xp = (CT)r.x; s[v][1].yp = (CT)r.y; s[v][1].zp = (CT)r.z; s[v][1].d = (CT)r.w;
        }
    }
}

// The couplings that other threads hold, through LDS.
template <typename CT>
__device__ __forceinline__ void t3_couplings_put(T3LDS<CT>& S, const T3Pos& t, const T3St<CT> (&s)[2][2]) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
        S.cy[q][t.e] = s[0][q].yp;
        S.cy[q][t.e + 256] = s[1][q].yp;
        S.cz[q][t.ec] = s[1][q].zp;
    }
}
template <typename CT>
__device__ __forceinline__ void t3_couplings_get(const T3LDS<CT>& S, const T3Pos& t, T3St<CT> (&s)[2][2]) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
        s[0][q].ym = t.rj >= 1 ? S.cy[q][t.e - 32] : CT(0);
        s[1][q].ym = t.rj >= 1 ? S.cy[q][t.e + 256 - 32] : CT(0);
        s[0][q].zm = t.rk >= 1 ? S.cz[q][t.ec - 256] : CT(0);
        s[1][q].zm = s[0][q].zp;
    }
}

// One colour of a thread's cells: on plane v the left or the right one.
// ON: in which rows and columns (ring: one cell inside the region; tile).
template <bool RING, typename CT>
__device__ __forceinline__ void t3_sweep(T3LDS<CT>& S, const T3Pos& t, bool even, CT (&x)[2][2], const CT (&b)[2][2], const T3St<CT> (&s)[2][2]) {
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const bool right = (t.left_odd == (v == 0)) == even;
        const CT xl = t3_left(t, x[v][1]), xr = t3_right(t, x[v][0]);   // all lanes: DPP reads the neighbours' registers
        const CT d = right ? s[v][1].d : s[v][0].d;
        const bool on = RING ? t.rr[v] && (right ? t.r1 : t.r0) : t.own;
        if (on && d >= CT(1e-30)) {
            const CT* X = S.x[right] + t.e + 256 * v;
            const CT xo = right ? x[v ^ 1][1] : x[v ^ 1][0];
            const CT up = X[32], dn = X[-32], fw = v ? X[256] : xo, bk = v ? xo : X[-256];
            const T3St<CT>&c0 = s[v][0], &c1 = s[v][1];
            const CT nb = (right ? c1.xp : c0.xp) * (right ? xr : x[v][1]) + (right ? c1.xm : c0.xm) * (right ? x[v][0] : xl)
                        + (right ? c1.yp : c0.yp) * up + (right ? c1.ym : c0.ym) * dn + (right ? c1.zp : c0.zp) * fw
                        + (right ? c1.zm : c0.zm) * bk;
            const CT n = mdiv<CT>((right ? b[v][1] : b[v][0]) + nb, d);
            if (right) x[v][1] = n;
            else x[v][0] = n;
        }
    }
}

// odd cells b / d; up: + 2 x_coarse on fluid cells
template <bool UP, typename CT>
__device__ __forceinline__ void t3_first(T3LDS<CT>& S, const T3Pos& t, CT (&x)[2][2], const CT (&b)[2][2], const T3St<CT> (&s)[2][2], CT c) {
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const bool odd = t.left_odd == ((v ^ q) == 0);
            CT n = (odd && s[v][q].d >= CT(1e-30)) ? mdiv<CT>(b[v][q] + CT(0), s[v][q].d) : CT(0);
            if (UP && s[v][q].d >= CT(0)) n = n + CT(2) * c;
            x[v][q] = n;
            S.x[q][t.e + 256 * v] = n;
        }
}
template <typename CT>
__device__ __forceinline__ void t3_put_even(T3LDS<CT>& S, const T3Pos& t, const CT (&x)[2][2]) {
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const bool right = t.left_odd == (v == 0);
        S.x[right][t.e + 256 * v] = right ? x[v][1] : x[v][0];
    }
}

// Down: forward sweep from x = 0, residual, restriction (b of the next level).
template <typename VB, typename C4>
__device__ __forceinline__ void d_t3_down(const VB* __restrict__ b, const C4* __restrict__ rec, const Geo& g, VB* __restrict__ bc, const Geo& cg,
                                          int tile, const int* skip) {
    using CT = typename CTOf<VB>::type;
    __shared__ T3LDS<CT> S;
    const int stop = skip ? *skip : 0;
    T3Pos t;
    t.init(g, tile);
    CT bv[2][2], x[2][2];
    T3St<CT> s[2][2];
    t3_load<VB, C4, CT>(b, rec, t, bv, s);
    if (stop) return;
#pragma unroll
    for (int v = 0; v < 2; v++) { s[v][0].xm = t3_left(t, s[v][1].xp); s[v][1].xm = s[v][0].xp; }
    t3_couplings_put<CT>(S, t, s);
    t3_first<false, CT>(S, t, x, bv, s, CT(0));
    __syncthreads();
    t3_couplings_get<CT>(S, t, s);
    // A neighbour has the other colour, so every value that the even cells
    // read was written before the barrier, and every one that they write is
    // read after the next.
    t3_sweep<true, CT>(S, t, true, x, bv, s);
    t3_put_even<CT>(S, t, x);
    __syncthreads();
    if (!t.own_wave) return;
    CT q[2][2];
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const CT xl = t3_left(t, x[v][1]), xr = t3_right(t, x[v][0]);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            q[v][c] = CT(0);
            const T3St<CT>& k = s[v][c];
            if (!t.own || !(k.d >= CT(0))) continue;
            const CT* X = S.x[c] + t.e + 256 * v;
            CT Ax = k.d * x[v][c] - k.xp * (c ? xr : x[v][1]) - k.xm * (c ? x[v][0] : xl);
            Ax = Ax - k.yp * X[32] - k.ym * X[-32];
            Ax = Ax - k.zp * (v ? X[256] : x[1][c]) - k.zm * (v ? x[0][c] : X[-256]);
            q[v][c] = bv[v][c] - Ax;
        }
    }
    // the coarse cell's children: these four and those of the row above, lane + 32
    CT sum = CT(0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const CT a0 = __shfl_down(q[0][c], 32, 64), a1 = __shfl_down(q[1][c], 32, 64);
        sum = sum + q[0][c] + q[1][c] + a0 + a1;
    }
    if (t.own && !(t.rj & 1)) {
        const int ic = (t.gi + 1) >> 1, jc = (t.gj + 1) >> 1, kc = (t.gk + 1) >> 1;
        if (ic <= cg.nx && jc <= cg.ny && kc <= cg.nz) bc[ic + jc * cg.sx + kc * cg.sy] = (VB)sum;
    }
}

// Up: x' = x0 + 2 x_coarse, reverse sweep.
template <typename VB, typename C4>
__device__ __forceinline__ void d_t3_up(const VB* __restrict__ b, const C4* __restrict__ rec, const Geo& g, const VB* __restrict__ xc, const Geo& cg,
                                        VB* __restrict__ xout, int tile, const int* skip) {
    using CT = typename CTOf<VB>::type;
    __shared__ T3LDS<CT> S;
    const int stop = skip ? *skip : 0;
    T3Pos t;
    t.init(g, tile);
    CT bv[2][2], x[2][2], c = CT(0);
    T3St<CT> s[2][2];
    {   // both planes of the thread have the same parent row
        const int ic = (t.gi + 1) >> 1, jc = (t.gj + 1) >> 1, kc = (t.gk + 1) >> 1;
        if ((t.in0[0] || t.in0[1]) && ic <= cg.nx && jc <= cg.ny && kc <= cg.nz) c = (CT)xc[ic + jc * cg.sx + kc * cg.sy];
    }
    t3_load<VB, C4, CT>(b, rec, t, bv, s);
    if (stop) return;
#pragma unroll
    for (int v = 0; v < 2; v++) { s[v][0].xm = t3_left(t, s[v][1].xp); s[v][1].xm = s[v][0].xp; }
    t3_couplings_put<CT>(S, t, s);
    t3_first<true, CT>(S, t, x, bv, s, c);
    __syncthreads();
    t3_couplings_get<CT>(S, t, s);
    t3_sweep<true, CT>(S, t, true, x, bv, s);      // even cells
    t3_put_even<CT>(S, t, x);
    __syncthreads();
    if (!t.own_wave) return;
    t3_sweep<false, CT>(S, t, false, x, bv, s);    // odd cells
#pragma unroll
    for (int v = 0; v < 2; v++)
        if (t.own && t.in0[v]) t2_put(xout + t.id[v], (VB)x[v][0], (VB)x[v][1], t.in1[v]);
}

template <typename VB, typename C4>
__global__ __launch_bounds__(T3_THREADS) void k_t3_down(const VB* __restrict__ b, const C4* __restrict__ rec, Geo g, VB* __restrict__ bc, Geo cg,
                                                        const int* skip) {
    const int t = tile_of_block();
    if (t < t3_tiles(g)) d_t3_down<VB, C4>(b, rec, g, bc, cg, t, skip);
}
template <typename VB, typename C4>
__global__ __launch_bounds__(T3_THREADS) void k_t3_up(const VB* __restrict__ b, const C4* __restrict__ rec, Geo g, const VB* __restrict__ xc, Geo cg,
                                                      VB* __restrict__ xout, const int* skip) {
    const int t = tile_of_block();
    if (t < t3_tiles(g)) d_t3_up<VB, C4>(b, rec, g, xc, cg, xout, t, skip);
}

}  // namespace uaamg
