// om_tend_centered.hip — z-marching, LDS-tiled tendency kernel for Centered(order=2) advection with a
// constant diffusivity or none, on three-dimensional grids with Periodic x and y and no immersed
// bottom (the default advection scheme, DNS).
//
// A block of 256 threads owns 32 × 8 columns and marches up a chunk of z levels.  The planes u, v,
// tracers at level k and w at k + 1, each with a one-cell ring, are staged in LDS (two slots, the
// next level's values loaded into registers while the current level is evaluated, one barrier per
// level); own-column values at k − 1 .. k + 1 and the z fluxes of the level's top face, which the next
// level takes as its bottom fluxes, stay in registers.  Horizontal fluxes are a few operations here,
// so each cell evaluates both its faces and no thread is spent on a tile's closing face.
//
// The flux formulas, their operand order and the tendency assembly are those of k_tendencies
// (om_kernels.hip); the two kernels give identically rounded results.  Latency and VALU issue bound
// it: 128³ FP64 with one tracer takes 48 µs (2.8 TB/s of its 134 MB in and out) where the
// thread-per-cell kernel, which tests topology, bottom and scheme at every face, takes 318 µs.
#include <hip/hip_runtime.h>

#include "om_batch.h"
#include "om_kernels.h"

namespace om {

constexpr int CNX = kCenteredX, CNY = kCenteredY;
constexpr int CPW = CNX + 2, CPR = CNY + 2, CPA = CPW * CPR;

template <class T, int NT> struct CenteredSmem {
    T u[2][CPA], v[2][CPA];
    T w[3][CPA];
    T c[NT > 0 ? NT : 1][2][CPA];
};

template <class T> struct TendCenteredArgs {
    Ctx<T> C;
    int kchunk, ntx;
};

template <class T, int NT> struct KTendCentered {
    static constexpr int kThreads = 256, kMinBlocks = 1;
    static constexpr bool kArgsInMemory = true;
    static __device__ __forceinline__ void run(const TendCenteredArgs<T> &A0, const Blk &B);
};

template <class T, int NT>
__device__ __forceinline__ void KTendCentered<T, NT>::run(const TendCenteredArgs<T> &A0, const Blk &B) {
    __shared__ CenteredSmem<T, NT> S;
    const ConstArgs<TendCenteredArgs<T>> args(A0);
    const TendCenteredArgs<T> &A = args.again();
    const Ctx<T> &C0 = A.C;
    const int kchunk = A.kchunk, ntx = A.ntx;
    const int tid = threadIdx.x;
    const int a = tid & (CNX - 1), b = tid / CNX;
    // work item → (z chunk, tile): the chunks of one tile are consecutive, tiles in row order
    const int item = xcd_work_item((int)B.x, (int)B.gx);
    const int nch = (C0.g.Nz + kchunk - 1) / kchunk;
    const int tile = item / nch, chunk = item - tile * nch;
    const int ty = tile / ntx, tx = tile - ty * ntx;
    const int i0 = tx * CNX, j0 = ty * CNY;
    const int k0 = chunk * kchunk, k1 = min(k0 + kchunk, C0.g.Nz);
    const int i = i0 + a, j = j0 + b;
    const bool cell = i < C0.g.Nx && j < C0.g.Ny;
    // (held inside the field: threads past its last halo point read a column nobody uses)
    const int ic = min(i, C0.g.Nx + C0.g.Hx - 1), jc = min(j, C0.g.Ny + C0.g.Hy - 1);
    const uint32_t colb = (uint32_t)(idx3(ic, jc, 0, C0.g.sy, C0.g.sz) * (int64_t)sizeof(T));
    const PlaneShare<T, CPW, CPR> ps(C0.g, i0, j0, 1, tid);
    auto P = [&](const T *p, int dx, int dy) -> T { return p[(b + 1 + dy) * CPW + (a + 1 + dx)]; };
    auto ldcol = [&](const Ctx<T> &C, const T *f, int k) -> T {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(f + (int64_t)k * C.g.sz) + colb);
    };

    T ru[2], rv[2], rw[2], rc[NT > 0 ? NT : 1][2];
    // u, v, tracers of level k and w of level k + 1
    auto load_level = [&](const Ctx<T> &C, int k) {
        const uint32_t o0 = ps.off0, o1 = ps.off1();
        ps.load(ru, ps.origin(C.s.U[0], C.g, i0, j0, 1, k), o0, o1);
        ps.load(rv, ps.origin(C.s.U[1], C.g, i0, j0, 1, k), o0, o1);
        ps.load(rw, ps.origin(C.s.U[2], C.g, i0, j0, 1, k + 1), o0, o1);
#pragma unroll
        for (int n = 0; n < NT; ++n) ps.load(rc[n], ps.origin(C.s.U[3 + n], C.g, i0, j0, 1, k), o0, o1);
    };
    const T half = T(0.5);
    T um, uc, vm, vc, wm, wc, cm[NT > 0 ? NT : 1], cc[NT > 0 ? NT : 1];   // own column at k − 1 and k
    T u1m, v1m;                                                          // u(i + 1) and v(j + 1) at k − 1
    {
        const Ctx<T> &C = args.again().C;
        um = ldcol(C, C.s.U[0], k0 - 1); uc = ldcol(C, C.s.U[0], k0);
        vm = ldcol(C, C.s.U[1], k0 - 1); vc = ldcol(C, C.s.U[1], k0);
        wm = ldcol(C, C.s.U[2], k0 - 1); wc = ldcol(C, C.s.U[2], k0);
#pragma unroll
        for (int n = 0; n < NT; ++n) { cm[n] = ldcol(C, C.s.U[3 + n], k0 - 1); cc[n] = ldcol(C, C.s.U[3 + n], k0); }
        const int ie = min(i + 1, C.g.Nx + C.g.Hx - 1), je = min(j + 1, C.g.Ny + C.g.Hy - 1);
        u1m = C.ld(C.s.U[0], ie, jc, k0 - 1);
        v1m = C.ld(C.s.U[1], ic, je, k0 - 1);
        ps.load(rw, ps.origin(C.s.U[2], C.g, i0, j0, 1, k0), ps.off0, ps.off1());
        ps.store(S.w[k0 % 3], rw, tid);
        load_level(C, k0);
    }
    // fluxes through the z face below level k: advective (F), viscous and diffusive (f; not yet times area)
    T Fu = T(0), Fv = T(0), Fw = T(0), Fc[NT > 0 ? NT : 1] = {}, fu = T(0), fv = T(0), fw = T(0), fc[NT > 0 ? NT : 1] = {};
    bool first = true;
    for (int k = k0; k < k1; ++k) {
        const int q = k & 1;
        T *const W1 = S.w[(k + 1) % 3];
        ps.store(S.u[q], ru, tid);
        ps.store(S.v[q], rv, tid);
        ps.store(W1, rw, tid);
#pragma unroll
        for (int n = 0; n < NT; ++n) ps.store(S.c[n][q], rc[n], tid);
        // one barrier: a slot is stored again two levels (w: three) later, after the next level's barrier
        __syncthreads();
        const Ctx<T> &C = args.again().C;
        const DevGrid<T> &g = C.g;
        const DevPhysics<T> &ph = C.ph;
        if (k + 1 < k1) load_level(C, k + 1);
        const T up = ldcol(C, C.s.U[0], k + 1), vp = ldcol(C, C.s.U[1], k + 1);
        T cp[NT > 0 ? NT : 1];
#pragma unroll
        for (int n = 0; n < NT; ++n) cp[n] = ldcol(C, C.s.U[3 + n], k + 1);
        const T *U = S.u[q], *V = S.v[q], *W0 = S.w[k % 3];
        const bool visc = ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY;
        const T Axc = g.dy * g.dzc[k], Ayc = g.dx * g.dzc[k], Axf = g.dy * g.dzf[k], Ayf = g.dx * g.dzf[k], Az = g.Az;
        const T idx = g.idx, idy = g.idy;
        const T nu = ph.c0, kap = ph.c1;
        // z fluxes of a face of level kk, from the w plane of that face and the column values around it
        auto zface = [&](const T *W, int kk, T u0, T u1, T v0, T v1, T &FU, T &FV, T &fU, T &fV) {
            const T wi = half * (P(W, -1, 0) + P(W, 0, 0)), wj = half * (P(W, 0, -1) + P(W, 0, 0));
            FU = Az * wi * (half * (u0 + u1));
            FV = Az * wj * (half * (v0 + v1));
            if (visc) {
                const T idzf = g.idzf[kk];
                const T dzu = (u1 - u0) * idzf, dxw = (P(W, 0, 0) - P(W, -1, 0)) * idx;
                const T dzv = (v1 - v0) * idzf, dyw = (P(W, 0, 0) - P(W, 0, -1)) * idy;
                const T S13 = half * (dzu + dxw), S23 = half * (dzv + dyw);
                fU = T(-2) * (nu * S13);
                fV = T(-2) * (nu * S23);
            }
        };
        auto zcentre = [&](int kk, T w0, T w1, T &FW, T &fW) {
            const T aw = half * (w0 + w1);
            FW = Az * aw * aw;
            if (visc) { const T dzw = (w1 - w0) * g.idzc[kk]; fW = T(-2) * (nu * dzw); }
        };
        auto zscalar = [&](int kk, T w, T c0, T c1, T &F, T &f) {
            F = (Az * w) * cen2<T>(c0, c1);
            if (visc) { const T dzc = (c1 - c0) * g.idzf[kk]; f = -kap * dzc; }
        };
        if (first) {
            first = false;
            zface(W0, k, um, uc, vm, vc, Fu, Fv, fu, fv);
            zcentre(k - 1, wm, wc, Fw, fw);
#pragma unroll
            for (int n = 0; n < NT; ++n) zscalar(k, wc, cm[n], cc[n], Fc[n], fc[n]);
        }
        const T wp = P(W1, 0, 0);
        T FuT, FvT, FwT, fuT = T(0), fvT = T(0), fwT = T(0);
        zface(W1, k + 1, uc, up, vc, vp, FuT, FvT, fuT, fvT);
        zcentre(k, wc, wp, FwT, fwT);
        const T u1 = P(U, 1, 0), v1 = P(V, 0, 1);
        if (cell) {
            const int64_t lo = (int64_t)k * g.sz;
            auto at = [&](T *f, int64_t shift) -> T & { return *reinterpret_cast<T *>(reinterpret_cast<char *>(f + lo + shift) + colb); };
            const T iVc = C.iVc(k), iVf = C.iVf(k);
            // strains at the ffc edges (i, j), (i, j + 1), (i + 1, j)
            auto s12 = [&](int dx, int dy) {
                const T dyu = (P(U, dx, dy) - P(U, dx, dy - 1)) * idy, dxv = (P(V, dx, dy) - P(V, dx - 1, dy)) * idx;
                return half * (dyu + dxv);
            };
            // advective fluxes of the horizontal edges
            auto F_Vu = [&](int dy) { const T vi = half * (P(V, -1, dy) + P(V, 0, dy)); return Ayc * vi * (half * (P(U, 0, dy - 1) + P(U, 0, dy))); };
            auto F_Uv = [&](int dx) { const T uj = half * (P(U, dx, -1) + P(U, dx, 0)); return Axc * uj * (half * (P(V, dx - 1, 0) + P(V, dx, 0))); };
            // ---------------- u
            {
                T G = T(0);
                const T ae = half * (uc + u1), aw = half * (P(U, -1, 0) + uc);
                const T Fe = Axc * ae * ae, Fwst = Axc * aw * aw;
                T sx = Fe - Fwst;
                T sy = F_Vu(1) - F_Vu(0);
                T sz = FuT - Fu;
                G -= iVc * ((sx + sy) + sz);
                if (ph.coriolis) {
                    const T Ac = Ayc;
                    auto q = [&](int dx, int dy) { return Ac * P(V, dx, dy); };   // (rounded before it is summed)
                    const T ca = half * (q(-1, 0) + q(0, 0));
                    const T cb = half * (q(-1, 1) + q(0, 1));
                    const T I = half * (ca + cb);
                    G += (half * (ph.f + ph.f)) * I * recip<T>(Ac);
                }
                if (ph.hydrostatic) {
                    const T d = C.s.dxpHY ? at(C.s.dxpHY, 0) : at(C.s.pHY, 0) - at(C.s.pHY, -1);
                    G -= d * idx;
                }
                if (visc) {
                    const T dxe = (u1 - uc) * idx, dxw = (uc - P(U, -1, 0)) * idx;
                    const T fe = T(-2) * (nu * dxe), fwst = T(-2) * (nu * dxw);
                    const T fn = T(-2) * (nu * s12(0, 1)), fs = T(-2) * (nu * s12(0, 0));
                    T vx = Axc * fe - Axc * fwst;
                    T vy = Ayc * fn - Ayc * fs;
                    T vz = Az * fuT - Az * fu;
                    G -= iVc * ((vx + vy) + vz);
                }
                at(C.s.Gn[0], 0) = G;
            }
            // ---------------- v
            {
                T G = T(0);
                const T an = half * (vc + v1), as = half * (P(V, 0, -1) + vc);
                const T Fn = Ayc * an * an, Fs = Ayc * as * as;
                T sx = F_Uv(1) - F_Uv(0);
                T sy = Fn - Fs;
                T sz = FvT - Fv;
                G -= iVc * ((sx + sy) + sz);
                if (ph.coriolis) {
                    const T Ac = Axc;
                    auto q = [&](int dx, int dy) { return Ac * P(U, dx, dy); };
                    const T ca = half * (q(0, -1) + q(1, -1));
                    const T cb = half * (q(0, 0) + q(1, 0));
                    const T I = half * (ca + cb);
                    G -= (half * (ph.f + ph.f)) * I * recip<T>(Ac);
                }
                if (ph.hydrostatic) {
                    const T d = C.s.dypHY ? at(C.s.dypHY, 0) : at(C.s.pHY, 0) - at(C.s.pHY, -g.sy);
                    G -= d * idy;
                }
                if (visc) {
                    const T fe = T(-2) * (nu * s12(1, 0)), fwst = T(-2) * (nu * s12(0, 0));
                    const T dyn = (v1 - vc) * idy, dys = (vc - P(V, 0, -1)) * idy;
                    const T fn = T(-2) * (nu * dyn), fs = T(-2) * (nu * dys);
                    T vx = Axc * fe - Axc * fwst;
                    T vy = Ayc * fn - Ayc * fs;
                    T vz = Az * fvT - Az * fv;
                    G -= iVc * ((vx + vy) + vz);
                }
                at(C.s.Gn[1], 0) = G;
            }
            // ---------------- w
            {
                T G = T(0);
                const T uk1 = half * (u1m + u1), uk0 = half * (um + uc);
                const T vk1 = half * (v1m + v1), vk0 = half * (vm + vc);
                const T Fe = Axf * uk1 * (half * (P(W0, 0, 0) + P(W0, 1, 0))), Fwst = Axf * uk0 * (half * (P(W0, -1, 0) + P(W0, 0, 0)));
                const T Fn = Ayf * vk1 * (half * (P(W0, 0, 0) + P(W0, 0, 1))), Fs = Ayf * vk0 * (half * (P(W0, 0, -1) + P(W0, 0, 0)));
                T sx = Fe - Fwst;
                T sy = Fn - Fs;
                T sz = FwT - Fw;
                G -= iVf * ((sx + sy) + sz);
                if (!ph.hydrostatic && ph.buoyancy != OM_BUOYANCY_NONE) {
                    T bm = T(0), b0 = T(0);
                    if (ph.buoyancy == OM_BUOYANCY_TRACER) {
#pragma unroll
                        for (int n = 0; n < NT; ++n) if (n == ph.b_tracer) { bm = cm[n]; b0 = cc[n]; }
                    } else {
                        T Tm = T(0), T0 = T(0), Sm = T(0), S0 = T(0);
#pragma unroll
                        for (int n = 0; n < NT; ++n) {
                            if (n == ph.T_tracer) { Tm = cm[n]; T0 = cc[n]; }
                            if (n == ph.S_tracer) { Sm = cm[n]; S0 = cc[n]; }
                        }
                        bm = ph.g * (ph.alpha * Tm - ph.beta * Sm);
                        b0 = ph.g * (ph.alpha * T0 - ph.beta * S0);
                    }
                    G += half * (bm + b0);
                }
                if (visc) {
                    const T idzf = g.idzf[k];
                    auto s13 = [&](T ua, T ub, int dx) {
                        const T dzu = (ub - ua) * idzf, dxw = (P(W0, dx, 0) - P(W0, dx - 1, 0)) * idx;
                        return half * (dzu + dxw);
                    };
                    auto s23 = [&](T va, T vb, int dy) {
                        const T dzv = (vb - va) * idzf, dyw = (P(W0, 0, dy) - P(W0, 0, dy - 1)) * idy;
                        return half * (dzv + dyw);
                    };
                    const T fe = T(-2) * (nu * s13(u1m, u1, 1)), fwst = T(-2) * (nu * s13(um, uc, 0));
                    const T fn = T(-2) * (nu * s23(v1m, v1, 1)), fs = T(-2) * (nu * s23(vm, vc, 0));
                    T vx = Axf * fe - Axf * fwst;
                    T vy = Ayf * fn - Ayf * fs;
                    T vz = Az * fwT - Az * fw;
                    G -= iVf * ((vx + vy) + vz);
                }
                at(C.s.Gn[2], 0) = G;
            }
        }
        // ---------------- tracers
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const T *Cn = S.c[n][q];
            T FT, fT = T(0);
            zscalar(k + 1, wp, cc[n], cp[n], FT, fT);
            if (cell) {
                const int64_t lo = (int64_t)k * g.sz;
                const T iVc = C.iVc(k);
                const T Fe = (Axc * u1) * cen2<T>(cc[n], P(Cn, 1, 0)), Fwst = (Axc * uc) * cen2<T>(P(Cn, -1, 0), cc[n]);
                const T Fn = (Ayc * v1) * cen2<T>(cc[n], P(Cn, 0, 1)), Fs = (Ayc * vc) * cen2<T>(P(Cn, 0, -1), cc[n]);
                T G = T(0);
                T sx = Fe - Fwst;
                T sy = Fn - Fs;
                T sz = FT - Fc[n];
                G -= iVc * ((sx + sy) + sz);
                if (visc) {
                    const T dxe = (P(Cn, 1, 0) - cc[n]) * idx, dxw = (cc[n] - P(Cn, -1, 0)) * idx;
                    const T dyn = (P(Cn, 0, 1) - cc[n]) * idy, dys = (cc[n] - P(Cn, 0, -1)) * idy;
                    const T fe = -kap * dxe, fwst = -kap * dxw, fn = -kap * dyn, fs = -kap * dys;
                    T vx = Axc * fe - Axc * fwst;
                    T vy = Ayc * fn - Ayc * fs;
                    T vz = Az * fT - Az * fc[n];
                    G -= iVc * ((vx + vy) + vz);
                }
                *reinterpret_cast<T *>(reinterpret_cast<char *>(C.s.Gn[3 + n] + lo) + colb) = G;
            }
            Fc[n] = FT;
            fc[n] = fT;
            cm[n] = cc[n];
            cc[n] = cp[n];
        }
        Fu = FuT; Fv = FvT; Fw = FwT;
        fu = fuT; fv = fvT; fw = fwT;
        um = uc; uc = up; vm = vc; vc = vp; wm = wc; wc = wp;
        u1m = u1; v1m = v1;
    }
}

template <class T> bool centered_tendencies_supported(const Ctx<T> &C) {
    const DevGrid<T> &g = C.g;
    return C.ph.advection == OM_ADV_CENTERED2 && (C.ph.closure == OM_CLOSURE_NONE || C.ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) &&
           g.tx == OM_PERIODIC && g.ty == OM_PERIODIC && (g.tz == OM_BOUNDED || g.tz == OM_PERIODIC) && g.Hx >= 1 && g.Hy >= 1 &&
           g.Hz >= 1 && C.ph.n_tracers <= 2 && !g.kbot;
}

template <class T> void launch_tend_centered(const Ctx<T> &C, int kchunk, hipStream_t st) {
    const DevGrid<T> &g = C.g;
    const int ntx = (g.Nx + CNX - 1) / CNX, nty = (g.Ny + CNY - 1) / CNY;
    if (kchunk < 1) kchunk = 1;
    const int nch = (g.Nz + kchunk - 1) / kchunk;
    const dim3 grid(ntx * nty * nch), blk(256);
    const TendCenteredArgs<T> A{C, kchunk, ntx};
    // (launched directly, not through a batch's recorder: batches hold WENO members only)
    switch (C.ph.n_tracers) {
        case 0: hipLaunchKernelGGL((k_one<KTendCentered<T, 0>, TendCenteredArgs<T>>), grid, blk, 0, st, A); break;
        case 1: hipLaunchKernelGGL((k_one<KTendCentered<T, 1>, TendCenteredArgs<T>>), grid, blk, 0, st, A); break;
        default: hipLaunchKernelGGL((k_one<KTendCentered<T, 2>, TendCenteredArgs<T>>), grid, blk, 0, st, A);
    }
}

#ifndef OM_ONLY_DOUBLE
template bool centered_tendencies_supported<float>(const Ctx<float> &);
template void launch_tend_centered<float>(const Ctx<float> &, int, hipStream_t);
#endif
#ifndef OM_ONLY_FLOAT
template bool centered_tendencies_supported<double>(const Ctx<double> &);
template void launch_tend_centered<double>(const Ctx<double> &, int, hipStream_t);
#endif

}  // namespace om
