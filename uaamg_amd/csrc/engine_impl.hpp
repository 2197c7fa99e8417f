// engine_impl.hpp -- Engine members defined out of the class, included by the
// sources that instantiate engines (engine_*.hip).
#pragma once
#include <algorithm>
#include <cstring>
#include <vector>
#include "engine.hpp"

namespace uaamg {

template <typename A, typename B>
__global__ void k_cast_all(const A* __restrict__ src, B* __restrict__ dst, long n) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x, s = (long)gridDim.x * blockDim.x;
    for (; t < n; t += s) dst[t] = (B)src[t];
}

template <int D, typename T, typename S, typename R>
void Engine<D, T, S, R>::cast_in_all(const double* src, T* dst) {
    long n = g0_.N;
    k_cast_all<double, T><<<(unsigned)std::min<long>((n + 255) / 256, 4096), 256, 0, stream_>>>(src, dst, n);
    HIPCHK(hipGetLastError());
}
template <int D, typename T, typename S, typename R>
void Engine<D, T, S, R>::cast_out_all(const T* src, double* dst) {
    long n = g0_.N;
    k_cast_all<T, double><<<(unsigned)std::min<long>((n + 255) / 256, 4096), 256, 0, stream_>>>(src, dst, n);
    HIPCHK(hipGetLastError());
}

template <int D, typename T, typename S, typename R>
void Engine<D, T, S, R>::allocate() {
    const int nl = nlevels();
    lv_.resize(nl);
    lv_[0].g = g0_;
    lv_[0].lc = lc0_;
    solid0_ = dalloc<uint8_t>(g0_.N);
    // kRowSlack: the row kernels load CPL consecutive cells per lane from a
    // clamped row start, up to CPL - 1 cells past the last ghost cell
    nbr0_ = dalloc<uint8_t>(N4_ + kRowSlack);
    count_ = dalloc<double>(1);
    ctrl_ = dalloc<Ctrl>(1);
    HIPCHK(hipHostMalloc((void**)&ctrl_host_, sizeof(Ctrl), hipHostMallocDefault));
    // the level-0 vectors in one allocation: r, z, p, Ap, x and, where the CG
    // passes are fused, the second p (GMG / AMG have it in any case, for x of
    // the coarse levels' way down) and in 3D with FP32 vectors the second r
    T** vec[] = {&r_, &z_, &p_, &Ap_, &x_, &p2_, &r2_};
    const int nv = pmv_on_ ? (FLATCG ? 6 : 7) : (gmg_ ? 6 : 5);
    const size_t stride = vec_stride(N4_, margin_);
    T* base = dalloc<T>(nv * stride);
    for (int q = 0; q < nv; q++) *vec[q] = base + q * stride + margin_;
    if (pmv_on_) partials_m_ = dalloc<double>(pmv_blocks_ + 64);
    long maxb = std::max<long>(lc0_.nblocks(), 2048);
    for (int l = 1; l < nl; l++) {
        Level& L = lv_[l];
        L.g = shape_[l];
        L.lc = cells_launch(L.g, D);
        L.b = dalloc<S>(L.g.N + kRowSlack); L.x = dalloc<S>(L.g.N + kRowSlack);
        L.mask = dalloc<uint8_t>(L.g.N);
        L.coef = dalloc<C4>(L.g.N + kRowSlack);
        L.ex = dalloc<S>(L.g.N);
        maxb = std::max(maxb, L.lc.nblocks());
    }
    maxb = std::max(maxb, fused_max_blocks());
    if (!FLATCG) maxb = std::max(maxb, (long)rows_blocks_);   // the FP64 row kernels write no partials
    partials_ = dalloc<double>(3 * maxb + 64);
    fused_ok_ = fused_supported();
    HIPCHK(hipStreamSynchronize(stream_));
}

template <int D, typename T, typename S, typename R>
void Engine<D, T, S, R>::release() {
    (void)hipStreamSynchronize(stream_);
    for (void* p : allocs_) (void)hipFree(p);
    allocs_.clear();
    if (ctrl_host_) (void)hipHostFree(ctrl_host_);
    ctrl_host_ = nullptr;
    if (hist_) (void)hipFree(hist_);
    hist_ = nullptr;
}

template <int D, typename T, typename S, typename R>
void Engine<D, T, S, R>::level_data(int level, uint8_t* solid, double* diag, double* cx, double* cy, double* cz, double* ex) {
    const Geo g = shape_[level];
    const long N = g.N;
    std::vector<uint8_t> m(N);
    std::vector<double> vx(N, 0.0), vy(N, 0.0), vz(N, 0.0), ve(N, 0.0), vd(N, 0.0);
    auto IX = [&](int i, int j, int k) { return (long)i + (long)j * g.sx + (long)k * g.sy; };
    const int klo = (D == 3) ? 1 : 0, khi = (D == 3) ? g.nz : 0;
    if (level == 0) {
        std::vector<uint8_t> nb(N);
        HIPCHK(hipMemcpyAsync(m.data(), solid0_, N, hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipMemcpyAsync(nb.data(), nbr0_, N, hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipStreamSynchronize(stream_));
        const Consts<double>& c = c0d_;
        for (int i = 1; i <= g.nx; i++)
            for (int j = 1; j <= g.ny; j++)
                for (int k = klo; k <= khi; k++) {
                    long id = IX(i, j, k);
                    if (!(nb[id] & NB_FLUID)) continue;
                    vx[id] = (nb[id] & NB_XP) ? c.idx2 : 0.0;
                    vy[id] = (nb[id] & NB_YP) ? c.idy2 : 0.0;
                    if (D == 3) vz[id] = (nb[id] & NB_ZP) ? c.idz2 : 0.0;
                    double e = 0.0;
                    if (c.wall[0] && i == 1) e += c.ex2[0];
                    if (c.wall[1] && i == g.nx) e += c.ex2[1];
                    if (c.wall[2] && j == 1) e += c.ex2[2];
                    if (c.wall[3] && j == g.ny) e += c.ex2[3];
                    if (D == 3) {
                        if (c.wall[4] && k == 1) e += c.ex2[4];
                        if (c.wall[5] && k == g.nz) e += c.ex2[5];
                    }
                    ve[id] = e;
                }
        for (int i = 1; i <= g.nx; i++)
            for (int j = 1; j <= g.ny; j++)
                for (int k = klo; k <= khi; k++) {
                    long id = IX(i, j, k);
                    if (!(nb[id] & NB_FLUID)) continue;
                    double d = (D == 3) ? vx[id] + vx[id - 1] + vy[id] + vy[id - g.sx] + vz[id] + vz[id - g.sy]
                                        : vx[id] + vx[id - 1] + vy[id] + vy[id - g.sx];
                    if (ve[id] != 0.0) d += ve[id];
                    vd[id] = d;
                }
    } else {
        const Level& L = lv_[level];
        std::vector<C4> cf(N);
        std::vector<S> exv(N);
        HIPCHK(hipMemcpyAsync(m.data(), L.mask, N, hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipMemcpyAsync(cf.data(), L.coef, N * sizeof(C4), hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipMemcpyAsync(exv.data(), L.ex, N * sizeof(S), hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipStreamSynchronize(stream_));
        for (int i = 1; i <= g.nx; i++)
            for (int j = 1; j <= g.ny; j++)
                for (int k = klo; k <= khi; k++) {
                    long id = IX(i, j, k);
                    vx[id] = (double)cf[id].x; vy[id] = (double)cf[id].y;
                    if (D == 3) vz[id] = (double)cf[id].z;
                    ve[id] = (double)exv[id];
                    // the record's diagonal as stored (solid cells carry -1, reported as 0)
                    vd[id] = m[id] ? 0.0 : (double)cf[id].w;
                }
    }
    if (solid) std::memcpy(solid, m.data(), N);
    if (diag) std::memcpy(diag, vd.data(), N * sizeof(double));
    if (cx) std::memcpy(cx, vx.data(), N * sizeof(double));
    if (cy) std::memcpy(cy, vy.data(), N * sizeof(double));
    if (cz && D == 3) std::memcpy(cz, vz.data(), N * sizeof(double));
    if (ex) std::memcpy(ex, ve.data(), N * sizeof(double));
}

}  // namespace uaamg
