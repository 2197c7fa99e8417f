// kernels_rows64.hpp -- level-0 V(1,1) kernels in 3D for FP64 vectors.
//
// The mapping of kernels_rows.hpp (whole rows or windows of two cells a lane,
// waves of 2 rows, a march along z), the arithmetic and order per cell of
// the per-pass and march kernels (and so the reference's smooth /
// restrictResidual / prolongateAdd, uaamg_preconditioner_3d.cpp:123-181), bit
// for bit: an FP64 solve of some ten iterations carries a changed last digit
// of one dot product into the ninth digit of its pressure.  So
//   * neighbour sums and residuals add x+, x-, y+, y-, z+, z- in that order (an
//     absent neighbour's value is 0), every fluid cell's residual is formed,
//     and a coarse cell adds its children x slowest, z fastest;
//   * divisions are divisions;
//   * the z sums are a pass of their own in the march kernel's order
//     (k_zsums_m3), which is cheaper than that kernel.
// A lane keeps d (< 0: not fluid) of its cells on four planes; the rows that
// waves share go through LDS, one slot per plane of the window and colour.
//
// Eight waves a workgroup, two per SIMD: with ten (168 VGPRs) the down kernel
// spilled 47 registers (36 us at 256 x 128 x 128, 13 at 128 x 64 x 64).  256 x 128
// x 128 (three windows): down 62 -> 26 us, up 70 -> 25 and 15 for the sums; 128 x
// 64 x 64: 25 -> 8.1, 30 -> 8.5 and 6.
#pragma once
#include "kernels_march.hpp"
#include "kernels_rows.hpp"

namespace uaamg {

constexpr int R64_NW = 8, R64_RW = 2, R64_CPL = 2;

struct Row64LDS {
    double d[64];                         // d per neighbour pattern, without walls
    double ex[4][2][R64_NW][2][64];       // [plane slot][0: odd, 1: even cells][wave][first / last row][lane]
};

template <bool WIN>
using Row64Thread = RowThread<R64_CPL, R64_NW, R64_RW, 2, false, WIN>;

// state of a lane's 2 x 2 cells on the four planes of the window
struct Row64Q { double X[4][2][2], D[4][2][2], B[4][2][2]; };

// d of the plane's cells (-1: not fluid)
template <bool WIN>
__device__ __forceinline__ void r64_diag(const uint8_t (&nb)[2][2], double (&d)[2][2], const Row64LDS& L, const Consts<double>& c,
                                         const Geo& g, const Row64Thread<WIN>& th, int k) {
    double v[2][2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int q = 0; q < 2; q++) v[t][q] = L.d[nb[t][q] >> 1];
    if (c.any_dirichlet) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const double e = wall_excess0<3, double>(c, g, th.i0 + q, th.jrow[t], k);
                if (e != 0.0) v[t][q] += e;
            }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int q = 0; q < 2; q++) d[t][q] = (nb[t][q] & NB_FLUID) ? v[t][q] : -1.0;
}

// The in-plane neighbours of cell (T, Q) of plane slot s: right, left, +y, -y.
struct Row64N { double xr, xl, yp, ym; };
template <int T, int Q, int s>
__device__ __forceinline__ Row64N r64_nb(const Row64Q& S, double edge, const Row64LDS& L, int kind, int w, int lane) {
    Row64N n;
    n.xr = Q == 0 ? S.X[s][T][1] : edge;
    n.xl = Q == 1 ? S.X[s][T][0] : edge;
    n.yp = T == 0 ? S.X[s][1][Q] : L.ex[s][kind][w < R64_NW - 1 ? w + 1 : R64_NW - 1][0][lane];
    n.ym = T == 1 ? S.X[s][0][Q] : L.ex[s][kind][w > 0 ? w - 1 : 0][1][lane];
    return n;
}

// one colour of plane slot s (sp, sm: the planes above and below); its first
// and last rows' cells go to LDS
template <int PAR, int s, int sp, int sm>
__device__ __forceinline__ void r64_colour(Row64Q& S, Row64LDS& L, const Consts<double>& c, int w, int lane) {
    sfor<2>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        constexpr int q = (PAR + t + s) & 1;          // the cell of this colour in the row ((q + t + s) & 1 == PAR)
        const double edge = q == 0 ? lane_from_left(S.X[s][t][1]) : lane_from_right(S.X[s][t][0]);
        const Row64N n = r64_nb<t, q, s>(S, edge, L, PAR ? 1 : 0, w, lane);   // neighbours have the other colour
        const double d = S.D[s][t][q];
        const double nb = c.idx2 * n.xr + c.idx2 * n.xl + c.idy2 * n.yp + c.idy2 * n.ym + c.idz2 * S.X[sp][t][q] + c.idz2 * S.X[sm][t][q];
        const double v = (S.B[s][t][q] + nb) / d;
        S.X[s][t][q] = d >= 1e-30 ? v : S.X[s][t][q];
    });
    if constexpr (PAR == 0)
        sfor<2>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            constexpr int q = (t + s) & 1;
            L.ex[s][1][w][t][lane] = S.X[s][t][q];
        });
}

__device__ __forceinline__ void r64_start(Row64LDS& L, Row64Q& S, const Consts<double>& c, const Geo& g) {
    for (int e = threadIdx.x; e < 64; e += R64_NW * 64) {
        Consts<double> k = c;
        k.any_dirichlet = 0;
        L.d[e] = msten0<3, double>((uint8_t)(NB_FLUID | (e << 1)), k, g, 2, 2, 2).d;
    }
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int q = 0; q < 2; q++) { S.X[s][t][q] = 0.0; S.D[s][t][q] = -1.0; S.B[s][t][q] = 0.0; }
    __syncthreads();
}

// Down: forward sweep from x = 0, residual, restriction.
template <bool WIN, typename VC>
__global__ __launch_bounds__(R64_NW * 64) void k_rows64_down0(const double* __restrict__ r, const uint8_t* __restrict__ nbr, Geo g,
                                                              Consts<double> c, RowGeo rg, VC* __restrict__ bc, Geo cg, const int* skip) {
    if (skip && *skip) return;
    const int tile = row_tile_of_block(rg, blockIdx.x);
    if (tile >= rg.ntiles) return;
    __shared__ Row64LDS L;
    Row64Thread<WIN> th;
    th.init(g, rg, tile);
    const int lane = th.lane, w = th.w;
    Row64Q S;
    double pfr[2][2][2], res[2][2];   // res: residuals of the odd plane of a pair, [x][y]
    uint8_t pfn[2][2][2];
    auto issue = [&](int slot, int P) {
        const int po = th.plane(g, P);
#pragma unroll
        for (int t = 0; t < 2; t++) row_load<2>(r, nbr, th.roff[t] + po, th.okx, pfr[slot][t], pfn[slot][t]);
    };
    issue(1, th.m0 - 2);
    issue(0, th.m0 - 1);
    r64_start(L, S, c, g);
    // plane P enters in slot s (P and s have the same parity)
    auto step = [&](auto sc, int P) {
        constexpr int s = decltype(sc)::value, s1 = (s + 3) & 3, s2 = (s + 2) & 3, s3 = (s + 1) & 3, PB = s & 1;
        r64_diag<WIN>(pfn[PB], S.D[s], L, c, g, th, P);
        sfor<2>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            constexpr int q = (1 + t + s) & 1;   // the odd cell
#pragma unroll
            for (int e = 0; e < 2; e++) { S.B[s][t][e] = (pfn[PB][t][e] & NB_FLUID) ? pfr[PB][t][e] : 0.0; S.X[s][t][e] = 0.0; }
            const double d = S.D[s][t][q], v = (S.B[s][t][q] + 0.0) / d;
            S.X[s][t][q] = d >= 1e-30 ? v : 0.0;
            L.ex[s][0][w][t][lane] = S.X[s][t][q];
        });
        issue(PB, min(P + 2, th.last + 2));   // past last + 2 (never used): the cached plane last + 2 again
        if (P - 1 >= th.m0 - 1) r64_colour<0, s1, s, s2>(S, L, c, w, lane);
        const int R = P - 2;
        if (R >= th.m0 && R <= th.last) {
            double q4[2][2];   // [x][y]
            sfor<2>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                const double el = lane_from_left(S.X[s2][t][1]), er = lane_from_right(S.X[s2][t][0]);
                sfor<2>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    constexpr int kind = ((q + t + s2) & 1) ? 1 : 0;      // an odd cell's neighbours are even
                    const Row64N n = r64_nb<t, q, s2>(S, q == 0 ? el : er, L, kind, w, lane);
                    const double d = S.D[s2][t][q];
                    double Ax = d * S.X[s2][t][q] - c.idx2 * n.xr - c.idx2 * n.xl;
                    Ax = Ax - c.idy2 * n.yp - c.idy2 * n.ym;
                    Ax = Ax - c.idz2 * S.X[s1][t][q] - c.idz2 * S.X[s3][t][q];
                    q4[q][t] = d >= 0.0 ? S.B[s2][t][q] - Ax : 0.0;
                });
            });
            if (R & 1) {
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int y = 0; y < 2; y++) res[x][y] = q4[x][y];
            } else {
                double sum = 0.0;
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int y = 0; y < 2; y++) { sum += res[x][y]; sum += q4[x][y]; }
                const int ic = (th.i0 + 1) >> 1, jc = (th.jrow[0] + 1) >> 1, kc = R >> 1;
                if (th.tile_row[0] && th.okw[0] && ic <= cg.nx && jc <= cg.ny && kc <= cg.nz)
                    bc[ic + jc * (int)cg.sx + kc * (int)cg.sy] = (VC)sum;
            }
        }
        __syncthreads();
    };
    for (int P = th.m0 - 2; P <= th.last + 2; P += 4) {
        step(IC<3>{}, P);
        if (P + 1 > th.last + 2) break;
        step(IC<0>{}, P + 1);
        if (P + 2 > th.last + 2) break;
        step(IC<1>{}, P + 2);
        if (P + 3 > th.last + 2) break;
        step(IC<2>{}, P + 3);
    }
}

// Up: x' = x0 + 2 x_coarse, reverse sweep, z.
template <bool WIN, typename VCX>
__global__ __launch_bounds__(R64_NW * 64) void k_rows64_up0(const double* __restrict__ r, const uint8_t* __restrict__ nbr, Geo g,
                                                            Consts<double> c, RowGeo rg, const VCX* __restrict__ xc, Geo cg,
                                                            double* __restrict__ z, const int* skip) {
    using RV = typename RowVec<2, double>::V;
    if (skip && *skip) return;
    const int tile = row_tile_of_block(rg, blockIdx.x);
    if (tile >= rg.ntiles) return;
    __shared__ Row64LDS L;
    Row64Thread<WIN> th;
    th.init(g, rg, tile);
    const int lane = th.lane, w = th.w;
    const int ic = (th.i0 + 1) >> 1, jc = (th.jrow[0] + 1) >> 1;   // both rows have the same parent row
    const bool cok = ic <= cg.nx && jc >= 1 && jc <= cg.ny;
    const int coff = min(ic, cg.nx + 1) + min(max(jc, 0), cg.ny + 1) * (int)cg.sx;
    Row64Q S;
    double pfr[2][2][2], pfx[2];
    uint8_t pfn[2][2][2];
    bool pcin[2];
    auto issue = [&](int slot, int P) {
        const int po = th.plane(g, P);
#pragma unroll
        for (int t = 0; t < 2; t++) row_load<2>(r, nbr, th.roff[t] + po, th.okx, pfr[slot][t], pfn[slot][t]);
        const int kc = (P + 1) >> 1;
        pcin[slot] = cok && kc >= 1 && kc <= cg.nz;
        pfx[slot] = (double)xc[coff + min(max(kc, 0), cg.nz + 1) * (int)cg.sy];
    };
    issue(1, th.m0 - 2);
    issue(0, th.m0 - 1);
    r64_start(L, S, c, g);
    auto step = [&](auto sc, int P) {
        constexpr int s = decltype(sc)::value, s1 = (s + 3) & 3, s2 = (s + 2) & 3, s3 = (s + 1) & 3, PB = s & 1;
        r64_diag<WIN>(pfn[PB], S.D[s], L, c, g, th, P);
        const double x2 = pcin[PB] ? 2.0 * pfx[PB] : 0.0;
        sfor<2>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            constexpr int q = (1 + t + s) & 1;   // the odd cell
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const bool fl = pfn[PB][t][e] & NB_FLUID;
                S.B[s][t][e] = fl ? pfr[PB][t][e] : 0.0;
                S.X[s][t][e] = fl ? 0.0 + x2 : 0.0;
            }
            const double d = S.D[s][t][q], v = (S.B[s][t][q] + 0.0) / d;
            if (d >= 1e-30) S.X[s][t][q] = v + x2;
            L.ex[s][0][w][t][lane] = S.X[s][t][q];
        });
        issue(PB, min(P + 2, th.last + 2));   // past last + 2 (never used): the cached plane last + 2 again
        if (P - 1 >= th.m0 - 1) r64_colour<0, s1, s, s2>(S, L, c, w, lane);
        const int R = P - 2;
        if (R >= th.m0 && R <= th.last) {
            r64_colour<1, s2, s1, s3>(S, L, c, w, lane);
            sfor<2>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                if (!th.tile_row[t]) return;
                double* out = z + th.roff[t] + R * (int)g.sy;
                if (th.okw[1]) *(RV*)out = RV{S.X[s2][t][0], S.X[s2][t][1]};
                else if (th.okw[0]) out[0] = S.X[s2][t][0];
            });
        }
        __syncthreads();
    };
    for (int P = th.m0 - 2; P <= th.last + 2; P += 4) {
        step(IC<3>{}, P);
        if (P + 1 > th.last + 2) break;
        step(IC<0>{}, P + 1);
        if (P + 2 > th.last + 2) break;
        step(IC<1>{}, P + 2);
        if (P + 3 > th.last + 2) break;
        step(IC<2>{}, P + 3);
    }
}

// sum z, sum r z, sum r over fluid cells with the cells, threads and order of
// k_up_m<3, true, RX, RY, PPT, true> (a tile of RX - 4 x RY - 4 cells and KC
// planes per workgroup, a thread's cells plane by plane).
template <int RX, int RY, int PPT>
__global__ __launch_bounds__(256) void k_zsums_m3(const double* __restrict__ z, const double* __restrict__ r, const uint8_t* __restrict__ nbr,
                                                  Geo g, int KC, const int* skip, double* partials) {
    if (skip && *skip) return;
    MPos<3, RX, RY, PPT> pos;
    const int m0 = blockIdx.z * KC + 1, last = min(m0 + KC - 1, g.nz);
    pos.init(g, blockIdx.x * (RX - 4) + 1, blockIdx.y * (RY - 4) + 1);
    double red[3] = {0.0, 0.0, 0.0};
    for (int k = m0; k <= last; k += 2) {   // two planes' loads at a time
        double zv[2][PPT], rv[2][PPT];
        bool on[2][PPT];
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int u = 0; u < PPT; u++) {
                on[v][u] = pos.r0[u] && pos.in[u] && k + v <= last;
                const long id = on[v][u] ? pos.off[u] + (long)(k + v) * g.sy : 0;
                zv[v][u] = z[id];
                rv[v][u] = r[id];
                on[v][u] = on[v][u] && (nbr[id] & NB_FLUID);
            }
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int u = 0; u < PPT; u++)
                if (on[v][u]) { red[0] += zv[v][u]; red[1] += rv[v][u] * zv[v][u]; red[2] += rv[v][u]; }
    }
    block_store<3>(red, partials);
}

}  // namespace uaamg
