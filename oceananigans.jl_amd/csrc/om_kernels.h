// om_kernels.h — device operators shared by the kernel sources, and the launcher interface
// used by the C-ABI host code.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <vector>

#include "om_internal.h"

namespace om {

// ----------------------------------------------------------------------------------------
// arithmetic helpers
// ----------------------------------------------------------------------------------------
// Approximate division for the WENO weights (the reference's BackendOptimizedDivision,
// src/Utils/newton_div.jl:57).  FP32: hardware reciprocal (≤1 ulp) times the numerator;
// FP64: IEEE division, so FP64 parity is not limited by it.
template <class T> __device__ __forceinline__ T wdiv(T a, T b);
template <> __device__ __forceinline__ float wdiv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <> __device__ __forceinline__ double wdiv<double>(double a, double b) { return a / b; }

// Unsigned division by a loop-invariant divisor d ≥ 1 with one multiply-high, a subtract and two
// shifts (Granlund & Montgomery, "Division by invariant integers using multiplication", 1994, §4).
struct FastDiv {
    uint32_t d, mul, s1, s2;
};
inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    FastDiv f;
    f.d = d;
    f.mul = (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
    f.s1 = l < 1 ? l : 1;
    f.s2 = l > 1 ? l - 1 : 0;
    return f;
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv &f) {
    const uint32_t t1 = __umulhi(f.mul, n);
    return (t1 + ((n - t1) >> f.s1)) >> f.s2;
}

// Reconstruction coefficients rounded to FT; the last entry of each tuple is 1 - Σ(others)
// evaluated in FT, as the reference builds them (reconstruction_coefficients.jl:74-76).
template <class T> struct RC {
    static constexpr T a0 = T(1.0 / 3), a1 = T(5.0 / 6), a2 = T(1) - (a0 + a1);      // WENO5 stencil 0
    static constexpr T b0 = T(-1.0 / 6), b1 = T(5.0 / 6), b2 = T(1) - (b0 + b1);     // stencil 1
    static constexpr T c0 = T(1.0 / 3), c1 = T(-7.0 / 6), c2 = T(1) - (c0 + c1);     // stencil 2
    static constexpr T d0 = T(0.5), d1 = T(1) - d0;                                   // WENO3 stencil 0
    static constexpr T e0 = T(-0.5), e1 = T(1) - e0;                                  // WENO3 stencil 1
    static constexpr T m1 = T(-1.0 / 12), s7 = T(7.0 / 12);
    static constexpr T q_p1 = m1, q_0 = s7, q_m1 = s7, q_m2 = T(1) - ((m1 + s7) + s7); // Centered(4)
    static constexpr T h_0 = T(0.5), h_m1 = T(1) - T(0.5);                            // Centered(2)
    static constexpr T C50 = T(3.0 / 10), C51 = T(3.0 / 5), C52 = T(1.0 / 10);
    static constexpr T C30 = T(2.0 / 3), C31 = T(1.0 / 3);
    static constexpr T eps = T(1e-8f);
};

// The reference evaluates the smoothness indicators, the WENO weighted sum and the Centered
// interpolants under @muladd (weno_interpolants.jl:265,279,516; centered_reconstruction.jl:56-62):
// a sum of products p₁ + p₂ + … + pₙ, evaluated left to right, becomes
// muladd(pₙ, muladd(…, muladd(p₂, p₁))), i.e. the first product rounded on its own and every later
// one fused into the running sum, and a product a·b·c splits as (a·b, c).  The generic templates
// below (the FP64 path: β, WENO3, Centered) spell these fused multiply-adds out and contract nothing else, so that
// identical inputs give the reference's rounding; weno5<double>'s weights and weighted sum alone
// round otherwise, and less (see there).  FP64 smoothness indicators on raw stencil
// values cancel heavily when the values carry a large offset, which makes the order observable.

// Smoothness quadratic form ψ₁(k₀ψ₁ + k₁ψ₂ + k₂ψ₃) + ψ₂(k₃ψ₂ + k₄ψ₃) + ψ₃ψ₃k₅
// (weno_interpolants.jl:172-174, 228-265)
template <class T> __device__ __forceinline__ T beta_q(T a, T b, T c, T k0, T k1, T k2, T k3, T k4, T k5) {
#pragma clang fp contract(off)
    const T s1 = fma(k2, c, fma(k1, b, k0 * a));
    const T s2 = fma(k4, c, k3 * b);
    return fma(c * c, k5, fma(b, s2, a * s1));
}

// 1/x for the FP64 weights: the hardware's estimate (2⁻²³ or better) and two Newton steps, 1 ulp
__device__ __forceinline__ double weight_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// WENO(order=5) value at face i from s0..s5 = ψ[i-3..i+2] (weno_interpolants.jl:348-354, 520-531)
template <class T> __device__ __forceinline__ T weno5(T s0, T s1, T s2, T s3, T s4, T s5, bool left);

// FP64: the smoothness indicators on raw values in the reference's order of operations (they cancel,
// so their rounding is visible), the Z weights with weight_rcp, and the weighted sum about the middle
// candidate, p_b + (α_a (p_a − p_b) + α_c (p_c − p_b)) / Σα.  The four IEEE divisions were 40 % of the
// instructions; without them 128³ tendencies take 208 instead of 250 µs.  Against extended precision
// (same indicators) the value's error is 0.6 - 0.95e-16 rms, 4.8e-16 at most, of the largest stencil value;
// dividing and summing ωₖ pₖ: 0.75 - 1.4e-16, 6.1e-16.
template <> __device__ __forceinline__ double weno5<double>(double s0, double s1, double s2, double s3, double s4, double s5, bool left) {
    typedef RC<double> K;
    const double t0 = left ? s0 : s5, t1 = left ? s1 : s4, t2 = left ? s2 : s3, t3 = left ? s3 : s2, t4 = left ? s4 : s1;
    const double ba = beta_q<double>(t2, t3, t4, 10.0, -31.0, 11.0, 25.0, -19.0, 4.0);
    const double bb = beta_q<double>(t1, t2, t3, 4.0, -13.0, 5.0, 13.0, -13.0, 4.0);
    const double bc = beta_q<double>(t0, t1, t2, 4.0, -19.0, 11.0, 25.0, -31.0, 10.0);
    const double tau = fabs(ba - bc);
    const double qa = tau * weight_rcp(ba + K::eps), qb = tau * weight_rcp(bb + K::eps), qc = tau * weight_rcp(bc + K::eps);
    // αₖ / C₅₁ (C₅₀ / C₅₁ = 1/2, C₅₂ / C₅₁ = 1/6)
    const double al0 = 0.5 * fma(qa, qa, 1.0), al1 = fma(qb, qb, 1.0), al2 = (1.0 / 6) * fma(qc, qc, 1.0);
    const double xa = t2 - t3, za = t4 - t3, xb = t1 - t2, xc = t0 - t1;
    const double da = fma(K::a2, za, fma(-K::b0, xb, (K::a0 + K::b2 - 1.0) * xa));
    const double dc = fma(K::c0, xc, fma(K::b2, xa, (1.0 - K::c2 - K::b0) * xb));
    const double pb = fma(K::b0, xb, fma(-K::b2, xa, t2));
    return fma(fma(al0, da, al2 * dc), weight_rcp((al0 + al1) + al2), pb);
}

// FP32 WENO(order=5): the same stencils, smoothness indicators on central-value-shifted values
// and Z weights, evaluated with fused multiply-adds and hardware reciprocals (≤ 1 ulp), and the
// weighted sum normalised once: Σ αₖ pₖ / Σ αₖ.  The reference's FP32 path rounds differently at
// the level of single ulps; FP32 results are held to the FP64 oracle within a stated tolerance,
// never bitwise, so the kernel spends its VALU budget on fewer instructions instead.
template <> __device__ __forceinline__ float weno5<float>(float s0, float s1, float s2, float s3, float s4, float s5, bool left) {
    typedef RC<float> K;
    // Mirror the stencil once: for either bias the three candidate stencils are then
    // a = (t2, t3, t4), b = (t1, t2, t3), c = (t0, t1, t2).
    const float t0 = left ? s0 : s5, t1 = left ? s1 : s4, t2 = left ? s2 : s3, t3 = left ? s3 : s2, t4 = left ? s4 : s1;
    // differences from each stencil's middle value (weno_interpolants.jl:276-281); neighbouring
    // stencils share them: b's right difference is −xa, c's is −xb
    const float xa = t2 - t3, za = t4 - t3, xb = t1 - t2, xc = t0 - t1;
    // The smoothness indicators and ε scaled by 1/4 (exact), which leaves every τ / (β + ε) as it
    // is: β_a/4 = 2.5 xa² + za (2.75 xa + za), β_b/4 = xb (xb − 1.25 xa) + xa²,
    // β_c/4 = 2.5 xb² + xc (xc − 2.75 xb), with xa² and xb² each formed once
    const float sa = xa * xa, sb = xb * xb;
    const float ba = fmaf(2.5f, sa, za * fmaf(2.75f, xa, za));
    const float bb = fmaf(xb, fmaf(-1.25f, xa, xb), sa);
    const float bc = fmaf(2.5f, sb, xc * fmaf(-2.75f, xb, xc));
    const float tau = fabsf(ba - bc);
    constexpr float eps4 = K::eps * 0.25f;
    const float qa = tau * __builtin_amdgcn_rcpf(ba + eps4);
    const float qb = tau * __builtin_amdgcn_rcpf(bb + eps4);
    const float qc = tau * __builtin_amdgcn_rcpf(bc + eps4);
    // the weights are normalised at the end, so the three αₖ may share any factor: here 1 / C₅₁,
    // which saves the middle stencil's multiplication (C₅₀ / C₅₁ = 1/2, C₅₂ / C₅₁ = 1/6)
    const float al0 = 0.5f * fmaf(qa, qa, 1.0f), al1 = fmaf(qb, qb, 1.0f), al2 = (1.0f / 6.0f) * fmaf(qc, qc, 1.0f);
    // candidate values: each stencil's coefficients sum to 1, so p = middle + k₀·x + k₂·z
    const float pa = fmaf(K::a0, xa, fmaf(K::a2, za, t3));
    const float pb = fmaf(K::b0, xb, fmaf(-K::b2, xa, t2));
    const float pc = fmaf(K::c0, xc, fmaf(-K::c2, xb, t1));
    const float num = fmaf(al0, pa, fmaf(al1, pb, al2 * pc));
    return num * __builtin_amdgcn_rcpf((al0 + al1) + al2);
}

// 1 / x: IEEE division in FP64 (the reference's rounding); the hardware reciprocal in FP32
template <class T> __device__ __forceinline__ T recip(T x) { return T(1) / x; }
template <> __device__ __forceinline__ float recip<float>(float x) { return __builtin_amdgcn_rcpf(x); }
// a / b: IEEE in FP64, a times the hardware reciprocal of b in FP32
template <class T> __device__ __forceinline__ T ft_div(T a, T b) { return a / b; }
template <> __device__ __forceinline__ float ft_div<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// WENO(order=3) smoothness ψ₁(ψ₁ − 2ψ₂) + ψ₂ψ₂·1 under @muladd
template <class T> __device__ __forceinline__ T beta2_q(T a, T b) {
#pragma clang fp contract(off)
    return fma(b * b, T(1), a * fma(T(-2), b, T(1) * a));
}

// WENO(order=3) value at face i from s0..s3 = ψ[i-2..i+1]
template <class T> __device__ __forceinline__ T weno3(T s0, T s1, T s2, T s3, bool left) {
    typedef RC<T> K;
    const T a0 = left ? s1 : s2, a1 = left ? s2 : s1;
    const T b0 = left ? s0 : s3, b1 = left ? s1 : s2;
    T ba, bb;
    if (sizeof(T) == 4) {
        const T da = a0 - a1, db = b0 - b1;
        ba = da * (T(1) * da + T(-2) * T(0)) + T(0);
        bb = db * (T(1) * db + T(-2) * T(0)) + T(0);
    } else {
        ba = beta2_q<T>(a0, a1);
        bb = beta2_q<T>(b0, b1);
    }
    const T tau = fabs(ba - bb);
    const T qa = wdiv<T>(tau, ba + K::eps), qb = wdiv<T>(tau, bb + K::eps);
    const T al0 = K::C30 * (T(1) + qa * qa), al1 = K::C31 * (T(1) + qb * qb);
    const T sinv = recip<T>(al0 + al1);
    return fma(al1 * sinv, K::e0 * b0 + K::e1 * b1, (al0 * sinv) * (K::d0 * a0 + K::d1 * a1));
}

// ℑ of four values, as the reference's nested two-point averages
template <class T> __device__ __forceinline__ T avg4(T a, T b, T c, T d) { return T(0.5) * (T(0.5) * (a + b) + T(0.5) * (c + d)); }
// FP32: ¼((a + b) + (c + d)), the same rounded value (scalings by powers of two are exact and
// commute with rounding, subnormal results aside) in two multiplications fewer
template <> __device__ __forceinline__ float avg4<float>(float a, float b, float c, float d) { return 0.25f * ((a + b) + (c + d)); }

// Centered(4) on offsets (−2, −1, 0, +1) from the face, under @muladd
template <class T> __device__ __forceinline__ T cen4(T m2, T m1, T z0, T p1) {
    typedef RC<T> K;
    return fma(K::q_p1, p1, fma(K::q_0, z0, fma(K::q_m1, m1, K::q_m2 * m2)));
}
// cen4 of four values that share one area factor A: in FP64 the reference's order,
// cen4(A·m2, A·m1, A·z0, A·p1); in FP32 the factor applied once to the interpolated value.
template <class T> __device__ __forceinline__ T acen4(T A, T m2, T m1, T z0, T p1) {
    if (sizeof(T) == 4) return A * cen4<T>(m2, m1, z0, p1);
    return cen4<T>(A * m2, A * m1, A * z0, A * p1);
}
// Centered(2) under @muladd (the same value as unfused: both products are exact halvings)
template <class T> __device__ __forceinline__ T cen2(T m1, T z0) {
    typedef RC<T> K;
    return fma(K::h_0, z0, K::h_m1 * m1);
}

// XCD-aware work order for a 1-D grid of nb blocks.  The dispatcher hands consecutive block ids to
// the 8 XCDs in turn, and each XCD has its own L2; this maps the blocks of one XCD onto one
// contiguous run of work items, so that tiles sharing halo planes share an L2.  A bijection on
// [0, nb): the first 8·⌊nb/8⌋ ids are redistributed, the remainder keeps its own id.
__device__ __forceinline__ int xcd_work_item(int id, int nb) {
    const int per = nb >> 3;
    if (id >= (per << 3)) return id;
    return (id & 7) * per + (id >> 3);
}

// A thread's share of a plane of R rows of W, staged into LDS by a 256-thread block: plane elements tid and
// tid + 256 (row-major, origin (i0 − h, j0 − h)).  The byte offset of the first from the plane origin
// is computed once per block and the second's follows from it (256 elements further on: a fixed
// number of rows and columns, and one row more where the column wraps), so staging a level costs one
// scalar origin per field and a load per element, and every load of a level can be issued before the
// first LDS store.  Offsets are held inside the level's plane, so no load is predicated: what the
// elements beyond the field's last halo point read is never used.
template <class T, int W, int R = W> struct PlaneShare {
    uint32_t off0, step, wrapstep, most;   // (the last three are the same for the whole block)
    bool wraps;
    __device__ __forceinline__ PlaneShare(const DevGrid<T> &g, int i0, int j0, int h, int tid) {
        static_assert(W * R >= 256 && W * R <= 512, "two elements per thread");
        constexpr uint32_t e = sizeof(T);
        const int y = tid / W, x = tid - y * W;
        most = (uint32_t)(g.sz - 1 - ((int64_t)(j0 - h + g.Hy) * g.sy + (i0 - h + g.Hx))) * e;
        step = ((uint32_t)(256 / W) * (uint32_t)g.sy + 256 % W) * e;
        wrapstep = step + ((uint32_t)g.sy - W) * e;
        off0 = min(((uint32_t)y * (uint32_t)g.sy + x) * e, most);
        wraps = x + 256 % W >= W;
    }
    // plane origin of field f at level k (uniform across the block)
    __device__ __forceinline__ static const char *origin(const T *f, const DevGrid<T> &g, int i0, int j0, int h, int k) {
        return reinterpret_cast<const char *>(f + idx3(i0 - h, j0 - h, k, g.sy, g.sz));
    }
    __device__ __forceinline__ uint32_t off1() const { return min(off0 + (wraps ? wrapstep : step), most); }
    __device__ __forceinline__ static void load(T (&v)[2], const char *base, uint32_t o0, uint32_t o1) {
        v[0] = *reinterpret_cast<const T *>(base + o0);
        if (threadIdx.x < W * R - 256) v[1] = *reinterpret_cast<const T *>(base + o1);
    }
    __device__ __forceinline__ static void store(T *dst, const T (&v)[2], int tid) {
        dst[tid] = v[0];
        if (tid < W * R - 256) dst[tid + 256] = v[1];
    }
};

// ----------------------------------------------------------------------------------------
// Immersed-bottom predicates (GridFittedBottom; src/Grids/inactive_node.jl:36-137,
// immersed_boundary_interface.jl), device indices (0-based).  A node at location (LX, LY, LZ)
// (0 Center, 1 Face) touches the cells i-a, j-b, k-c for a ≤ LX, b ≤ LY, c ≤ LZ: it is inactive
// when all of them are and peripheral when any of them is (the reference's recursion, unrolled).
// ----------------------------------------------------------------------------------------
template <class T> struct IB {
    const DevGrid<T> &g;
    __device__ __forceinline__ explicit IB(const DevGrid<T> &gg) : g(gg) {}
    __device__ __forceinline__ bool on() const { return g.kbot != nullptr; }
    __device__ __forceinline__ bool outside(int k) const { return g.tz == OM_BOUNDED && (k < 0 || k >= g.Nz); }
    __device__ __forceinline__ int column(int i, int j) const { return (i + kBottomMargin) + (g.Nx + 2 * kBottomMargin) * (j + kBottomMargin); }
    __device__ __forceinline__ bool immersed(int i, int j, int k) const { return g.kbot && k < g.kbot_wide[column(i, j)]; }
    __device__ __forceinline__ bool inactive_cell(int i, int j, int k) const { return immersed(i, j, k) || outside(k); }
    template <int LX, int LY, int LZ> __device__ __forceinline__ bool all_inactive(int i, int j, int k, bool under) const {
        bool r = true;
#pragma unroll
        for (int a = 0; a <= LX; ++a)
#pragma unroll
            for (int b = 0; b <= LY; ++b)
#pragma unroll
                for (int c = 0; c <= LZ; ++c) r = r && (under ? outside(k - c) : inactive_cell(i - a, j - b, k - c));
        return r;
    }
    template <int LX, int LY, int LZ> __device__ __forceinline__ bool any_inactive(int i, int j, int k, bool under) const {
        bool r = false;
#pragma unroll
        for (int a = 0; a <= LX; ++a)
#pragma unroll
            for (int b = 0; b <= LY; ++b)
#pragma unroll
                for (int c = 0; c <= LZ; ++c) r = r || (under ? outside(k - c) : inactive_cell(i - a, j - b, k - c));
        return r;
    }
    // immersed_inactive_node / immersed_peripheral_node: on the immersed grid but not on the underlying one
    template <int LX, int LY, int LZ> __device__ __forceinline__ bool iin(int i, int j, int k) const {
        return on() && all_inactive<LX, LY, LZ>(i, j, k, false) && !all_inactive<LX, LY, LZ>(i, j, k, true);
    }
    template <int LX, int LY, int LZ> __device__ __forceinline__ bool iper(int i, int j, int k) const {
        return on() && any_inactive<LX, LY, LZ>(i, j, k, false) && !any_inactive<LX, LY, LZ>(i, j, k, true);
    }
    // conditional δ between two points of one location (conditional_differences.jl:15-44)
    template <int LX, int LY, int LZ> __device__ __forceinline__ bool zd(int i1, int j1, int k1, int i2, int j2, int k2) const {
        return on() && (iin<LX, LY, LZ>(i1, j1, k1) || iin<LX, LY, LZ>(i2, j2, k2));
    }
    // near_{x,y,z}_immersed_boundary (immersed_advective_fluxes.jl:127-215) for buffers 3 (x) and 2 (y): any
    // inactive node among the 2·buffer stencil points; cell centres for a face interpolation point
    // (cs = false), faces along d for a centre interpolation point (cs = true).  A column's
    // inactive levels are those below its bottom and those outside a Bounded z, so along x and y the answer
    // is a comparison with the window's highest bottom (DevGrid::near_xy; a face is inactive below the
    // lower of its two bottoms), and along z the window's ends decide.  Looking up every point was most
    // of what the fix-up launches issued: with the tables (and kFixX's tiles) 487 → 155 µs for the
    // tendencies and 103 → 41 µs for the closure of the 256 × 256 × 128 seamount.
    struct Near {
        bool b3, b2;
    };
    __device__ __forceinline__ Near near(int d, bool cs, int i, int j, int k) const {
        if (d == 2) {
            const int kb = g.kbot_wide[column(i, j)];
            auto any = [&](int buffer) { return k - buffer + (cs ? 1 : 0) < kb || (g.tz == OM_BOUNDED && k + buffer - 1 >= g.Nz); };
            return Near{any(3), any(2)};
        }
        const int2 m = g.near_xy[4 * (int64_t)column(i, j) + 2 * d + (cs ? 1 : 0)];
        const bool out = outside(k);
        return Near{k < m.x || out, k < m.y || out};
    }
    // buffer chain WENO5 (0) → WENO3 (1) → Centered(2) (2); `topo` is the choice without an immersed boundary
    __device__ __forceinline__ int bsch(int d, bool cs, int i, int j, int k, int topo) const {
        if (!on()) return topo;
        const Near n = near(d, cs, i, j, k);
        return !n.b3 ? 0 : (n.b2 ? 2 : 1);
    }
    // advecting velocity: Centered(4) (true) or Centered(2) (false)
    __device__ __forceinline__ bool s4(int d, bool cs, int i, int j, int k, bool topo) const {
        if (!on()) return topo;
        return !near(d, cs, i, j, k).b3;
    }
};

// ----------------------------------------------------------------------------------------
// Context: grid + state + physics with the reference's operators as member functions
// ----------------------------------------------------------------------------------------
template <class T> struct Ctx {
    DevGrid<T> g;
    StateView<T> s;
    DevPhysics<T> ph;

    __device__ __forceinline__ int64_t at(int i, int j, int k) const { return idx3(i, j, k, g.sy, g.sz); }
    __device__ __forceinline__ T ld(const T *f, int i, int j, int k) const { return f[at(i, j, k)]; }
    __device__ __forceinline__ bool flx() const { return g.tx == OM_FLAT; }
    __device__ __forceinline__ bool fly() const { return g.ty == OM_FLAT; }
    __device__ __forceinline__ bool flz() const { return g.tz == OM_FLAT; }
    __device__ __forceinline__ bool bz() const { return g.tz == OM_BOUNDED; }

    // metric operators (area at z-Center / z-Face, volume)
    __device__ __forceinline__ T Axc(int k) const { return g.dy * g.dzc[k]; }
    __device__ __forceinline__ T Axf(int k) const { return g.dy * g.dzf[k]; }
    __device__ __forceinline__ T Ayc(int k) const { return g.dx * g.dzc[k]; }
    __device__ __forceinline__ T Ayf(int k) const { return g.dx * g.dzf[k]; }
    __device__ __forceinline__ T iVc(int k) const { return recip<T>(g.Az * g.dzc[k]); }
    __device__ __forceinline__ T iVf(int k) const { return recip<T>(g.Az * g.dzf[k]); }

    // z boundary switching: 0 = 5th-order (or Centered4), 1 = 3rd-order, 2 = Centered2
    __device__ __forceinline__ int zb_face(int k) const {
        if (!bz()) return 0;
        const int kr = k + 1, N = g.Nz;
        return (kr >= 4 && kr <= N - 2) ? 0 : ((kr >= 3 && kr <= N - 1) ? 1 : 2);
    }
    __device__ __forceinline__ int zb_center(int k) const {
        if (!bz()) return 0;
        const int kr = k + 1, N = g.Nz;
        return (kr >= 3 && kr <= N - 2) ? 0 : ((kr >= 2 && kr <= N - 1) ? 1 : 2);
    }
    __device__ __forceinline__ bool zs4_face(int k) const { const int kr = k + 1; return !bz() || (kr >= 4 && kr <= g.Nz - 2); }
    __device__ __forceinline__ bool zs4_center(int k) const { const int kr = k + 1; return !bz() || (kr >= 3 && kr <= g.Nz - 2); }

    // ---- biased reconstructions of field f at faces with scheme sch (0 WENO5, 1 WENO3, 2 Centered(2));
    // x and y switch only next to an immersed bottom
    __device__ __forceinline__ T bx_s(const T *f, int i, int j, int k, bool left, int sch) const {
        if (sch == 0) return weno5<T>(ld(f, i - 3, j, k), ld(f, i - 2, j, k), ld(f, i - 1, j, k), ld(f, i, j, k), ld(f, i + 1, j, k), ld(f, i + 2, j, k), left);
        if (sch == 1) return weno3<T>(ld(f, i - 2, j, k), ld(f, i - 1, j, k), ld(f, i, j, k), ld(f, i + 1, j, k), left);
        return cen2<T>(ld(f, i - 1, j, k), ld(f, i, j, k));
    }
    __device__ __forceinline__ T by_s(const T *f, int i, int j, int k, bool left, int sch) const {
        if (sch == 0) return weno5<T>(ld(f, i, j - 3, k), ld(f, i, j - 2, k), ld(f, i, j - 1, k), ld(f, i, j, k), ld(f, i, j + 1, k), ld(f, i, j + 2, k), left);
        if (sch == 1) return weno3<T>(ld(f, i, j - 2, k), ld(f, i, j - 1, k), ld(f, i, j, k), ld(f, i, j + 1, k), left);
        return cen2<T>(ld(f, i, j - 1, k), ld(f, i, j, k));
    }
    // z face k with scheme s (stencil centred on face k)
    __device__ __forceinline__ T bz_s(const T *f, int i, int j, int k, bool left, int sch) const {
        if (sch == 0) return weno5<T>(ld(f, i, j, k - 3), ld(f, i, j, k - 2), ld(f, i, j, k - 1), ld(f, i, j, k), ld(f, i, j, k + 1), ld(f, i, j, k + 2), left);
        if (sch == 1) return weno3<T>(ld(f, i, j, k - 2), ld(f, i, j, k - 1), ld(f, i, j, k), ld(f, i, j, k + 1), left);
        return cen2<T>(ld(f, i, j, k - 1), ld(f, i, j, k));
    }

    // ================= momentum advective fluxes (upwind_biased_advective_fluxes.jl:23-93); on an
    // immersed grid they vanish on the immersed periphery (immersed_advective_fluxes.jl:19-70) and the
    // interpolation order drops next to immersed cells (immersed_advective_fluxes.jl:127-215)
    __device__ __forceinline__ T F_Uu(int i, int j, int k) const {  // ccc
        const T *u = s.U[0];
        if (ph.advection == OM_ADV_CENTERED2) { T a = T(0.5) * (ld(u, i, j, k) + ld(u, i + 1, j, k)); return Axc(k) * a * a; }
        const IB<T> ib(g);
        if (ib.template iper<0, 0, 0>(i, j, k)) return T(0);
        const T A = Axc(k);
        const T ut = ib.s4(0, true, i, j, k, true) ? cen4<T>(A * ld(u, i - 1, j, k), A * ld(u, i, j, k), A * ld(u, i + 1, j, k), A * ld(u, i + 2, j, k))
                                                  : cen2<T>(A * ld(u, i, j, k), A * ld(u, i + 1, j, k));
        return ut * bx_s(u, i + 1, j, k, ut > T(0), ib.bsch(0, true, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Vu(int i, int j, int k) const {  // ffc
        if (fly()) return T(0);
        const T *u = s.U[0], *v = s.U[1];
        if (ph.advection == OM_ADV_CENTERED2) {
            T vi = flx() ? ld(v, i, j, k) : T(0.5) * (ld(v, i - 1, j, k) + ld(v, i, j, k));
            return Ayc(k) * vi * (T(0.5) * (ld(u, i, j - 1, k) + ld(u, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<1, 1, 0>(i, j, k)) return T(0);
        const T A = Ayc(k);
        const T vt = flx() ? A * ld(v, i, j, k)
                           : (ib.s4(0, false, i, j, k, true) ? cen4<T>(A * ld(v, i - 2, j, k), A * ld(v, i - 1, j, k), A * ld(v, i, j, k), A * ld(v, i + 1, j, k))
                                                             : cen2<T>(A * ld(v, i - 1, j, k), A * ld(v, i, j, k)));
        return vt * by_s(u, i, j, k, vt > T(0), ib.bsch(1, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Wu(int i, int j, int k) const {  // fcf
        if (flz()) return T(0);
        const T *u = s.U[0], *w = s.U[2];
        if (ph.advection == OM_ADV_CENTERED2) {
            T wi = flx() ? ld(w, i, j, k) : T(0.5) * (ld(w, i - 1, j, k) + ld(w, i, j, k));
            return g.Az * wi * (T(0.5) * (ld(u, i, j, k - 1) + ld(u, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<1, 0, 1>(i, j, k)) return T(0);
        const T A = g.Az;
        const T wt = flx() ? A * ld(w, i, j, k)
                           : (ib.s4(0, false, i, j, k, true) ? cen4<T>(A * ld(w, i - 2, j, k), A * ld(w, i - 1, j, k), A * ld(w, i, j, k), A * ld(w, i + 1, j, k))
                                                             : cen2<T>(A * ld(w, i - 1, j, k), A * ld(w, i, j, k)));
        return wt * bz_s(u, i, j, k, wt > T(0), ib.bsch(2, false, i, j, k, zb_face(k)));
    }
    __device__ __forceinline__ T F_Uv(int i, int j, int k) const {  // ffc
        if (flx()) return T(0);
        const T *u = s.U[0], *v = s.U[1];
        if (ph.advection == OM_ADV_CENTERED2) {
            T uj = fly() ? ld(u, i, j, k) : T(0.5) * (ld(u, i, j - 1, k) + ld(u, i, j, k));
            return Axc(k) * uj * (T(0.5) * (ld(v, i - 1, j, k) + ld(v, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<1, 1, 0>(i, j, k)) return T(0);
        const T A = Axc(k);
        const T ut = fly() ? A * ld(u, i, j, k)
                           : (ib.s4(1, false, i, j, k, true) ? cen4<T>(A * ld(u, i, j - 2, k), A * ld(u, i, j - 1, k), A * ld(u, i, j, k), A * ld(u, i, j + 1, k))
                                                             : cen2<T>(A * ld(u, i, j - 1, k), A * ld(u, i, j, k)));
        return ut * bx_s(v, i, j, k, ut > T(0), ib.bsch(0, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Vv(int i, int j, int k) const {  // ccc
        const T *v = s.U[1];
        if (ph.advection == OM_ADV_CENTERED2) { T a = T(0.5) * (ld(v, i, j, k) + ld(v, i, j + 1, k)); return Ayc(k) * a * a; }
        const IB<T> ib(g);
        if (ib.template iper<0, 0, 0>(i, j, k)) return T(0);
        const T A = Ayc(k);
        const T vt = ib.s4(1, true, i, j, k, true) ? cen4<T>(A * ld(v, i, j - 1, k), A * ld(v, i, j, k), A * ld(v, i, j + 1, k), A * ld(v, i, j + 2, k))
                                                  : cen2<T>(A * ld(v, i, j, k), A * ld(v, i, j + 1, k));
        return vt * by_s(v, i, j + 1, k, vt > T(0), ib.bsch(1, true, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Wv(int i, int j, int k) const {  // cff
        if (flz()) return T(0);
        const T *v = s.U[1], *w = s.U[2];
        if (ph.advection == OM_ADV_CENTERED2) {
            T wj = fly() ? ld(w, i, j, k) : T(0.5) * (ld(w, i, j - 1, k) + ld(w, i, j, k));
            return g.Az * wj * (T(0.5) * (ld(v, i, j, k - 1) + ld(v, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<0, 1, 1>(i, j, k)) return T(0);
        const T A = g.Az;
        const T wt = fly() ? A * ld(w, i, j, k)
                           : (ib.s4(1, false, i, j, k, true) ? cen4<T>(A * ld(w, i, j - 2, k), A * ld(w, i, j - 1, k), A * ld(w, i, j, k), A * ld(w, i, j + 1, k))
                                                             : cen2<T>(A * ld(w, i, j - 1, k), A * ld(w, i, j, k)));
        return wt * bz_s(v, i, j, k, wt > T(0), ib.bsch(2, false, i, j, k, zb_face(k)));
    }
    __device__ __forceinline__ T F_Uw(int i, int j, int k) const {  // fcf
        if (flx()) return T(0);
        const T *u = s.U[0], *w = s.U[2];
        if (ph.advection == OM_ADV_CENTERED2) {
            T uk = flz() ? ld(u, i, j, k) : T(0.5) * (ld(u, i, j, k - 1) + ld(u, i, j, k));
            return Axf(k) * uk * (T(0.5) * (ld(w, i - 1, j, k) + ld(w, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<1, 0, 1>(i, j, k)) return T(0);
        T ut;
        if (flz()) ut = Axc(k) * ld(u, i, j, k);
        else if (ib.s4(2, false, i, j, k, zs4_face(k)))
            ut = cen4<T>(Axc(k - 2) * ld(u, i, j, k - 2), Axc(k - 1) * ld(u, i, j, k - 1), Axc(k) * ld(u, i, j, k), Axc(k + 1) * ld(u, i, j, k + 1));
        else ut = cen2<T>(Axc(k - 1) * ld(u, i, j, k - 1), Axc(k) * ld(u, i, j, k));
        return ut * bx_s(w, i, j, k, ut > T(0), ib.bsch(0, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Vw(int i, int j, int k) const {  // cff
        if (fly()) return T(0);
        const T *v = s.U[1], *w = s.U[2];
        if (ph.advection == OM_ADV_CENTERED2) {
            T vk = flz() ? ld(v, i, j, k) : T(0.5) * (ld(v, i, j, k - 1) + ld(v, i, j, k));
            return Ayf(k) * vk * (T(0.5) * (ld(w, i, j - 1, k) + ld(w, i, j, k)));
        }
        const IB<T> ib(g);
        if (ib.template iper<0, 1, 1>(i, j, k)) return T(0);
        T vt;
        if (flz()) vt = Ayc(k) * ld(v, i, j, k);
        else if (ib.s4(2, false, i, j, k, zs4_face(k)))
            vt = cen4<T>(Ayc(k - 2) * ld(v, i, j, k - 2), Ayc(k - 1) * ld(v, i, j, k - 1), Ayc(k) * ld(v, i, j, k), Ayc(k + 1) * ld(v, i, j, k + 1));
        else vt = cen2<T>(Ayc(k - 1) * ld(v, i, j, k - 1), Ayc(k) * ld(v, i, j, k));
        return vt * by_s(w, i, j, k, vt > T(0), ib.bsch(1, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_Ww(int i, int j, int k) const {  // ccc (centre k uses the face k+1 stencils)
        if (flz()) return T(0);
        const T *w = s.U[2];
        if (ph.advection == OM_ADV_CENTERED2) { T a = T(0.5) * (ld(w, i, j, k) + ld(w, i, j, k + 1)); return g.Az * a * a; }
        const IB<T> ib(g);
        if (ib.template iper<0, 0, 0>(i, j, k)) return T(0);
        const T A = g.Az;
        const T wt = ib.s4(2, true, i, j, k, zs4_center(k)) ? cen4<T>(A * ld(w, i, j, k - 1), A * ld(w, i, j, k), A * ld(w, i, j, k + 1), A * ld(w, i, j, k + 2))
                                                           : cen2<T>(A * ld(w, i, j, k), A * ld(w, i, j, k + 1));
        return wt * bz_s(w, i, j, k + 1, wt > T(0), ib.bsch(2, true, i, j, k, zb_center(k)));
    }
    // ================= tracer advective fluxes (upwind_biased_advective_fluxes.jl:99-121)
    __device__ __forceinline__ T F_cx(const T *c, int i, int j, int k) const {
        const T ui = ld(s.U[0], i, j, k);
        if (ph.advection == OM_ADV_CENTERED2) return (Axc(k) * ui) * cen2<T>(ld(c, i - 1, j, k), ld(c, i, j, k));
        const IB<T> ib(g);
        if (ib.template iper<1, 0, 0>(i, j, k)) return T(0);
        return Axc(k) * ui * bx_s(c, i, j, k, ui > T(0), ib.bsch(0, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_cy(const T *c, int i, int j, int k) const {
        const T vj = ld(s.U[1], i, j, k);
        if (ph.advection == OM_ADV_CENTERED2) return (Ayc(k) * vj) * cen2<T>(ld(c, i, j - 1, k), ld(c, i, j, k));
        const IB<T> ib(g);
        if (ib.template iper<0, 1, 0>(i, j, k)) return T(0);
        return Ayc(k) * vj * by_s(c, i, j, k, vj > T(0), ib.bsch(1, false, i, j, k, 0));
    }
    __device__ __forceinline__ T F_cz(const T *c, int i, int j, int k) const {
        const T wk = ld(s.U[2], i, j, k);
        if (ph.advection == OM_ADV_CENTERED2) return (g.Az * wk) * cen2<T>(ld(c, i, j, k - 1), ld(c, i, j, k));
        const IB<T> ib(g);
        if (ib.template iper<0, 0, 1>(i, j, k)) return T(0);
        return g.Az * wk * bz_s(c, i, j, k, wk > T(0), ib.bsch(2, false, i, j, k, zb_face(k)));
    }

    // ================= gradients (velocity_tracer_gradients.jl:6-18)
    // conditional δ next to an immersed bottom (conditional_differences.jl:15-44)
    __device__ __forceinline__ T dx_u(int i, int j, int k) const { return flx() || IB<T>(g).template zd<1, 0, 0>(i, j, k, i + 1, j, k) ? T(0) : (ld(s.U[0], i + 1, j, k) - ld(s.U[0], i, j, k)) * g.idx; }
    __device__ __forceinline__ T dy_v(int i, int j, int k) const { return fly() || IB<T>(g).template zd<0, 1, 0>(i, j, k, i, j + 1, k) ? T(0) : (ld(s.U[1], i, j + 1, k) - ld(s.U[1], i, j, k)) * g.idy; }
    __device__ __forceinline__ T dz_w(int i, int j, int k) const { return flz() || IB<T>(g).template zd<0, 0, 1>(i, j, k, i, j, k + 1) ? T(0) : (ld(s.U[2], i, j, k + 1) - ld(s.U[2], i, j, k)) * g.idzc[k]; }
    __device__ __forceinline__ T dx_v(int i, int j, int k) const { return flx() || IB<T>(g).template zd<0, 1, 0>(i, j, k, i - 1, j, k) ? T(0) : (ld(s.U[1], i, j, k) - ld(s.U[1], i - 1, j, k)) * g.idx; }
    __device__ __forceinline__ T dx_w(int i, int j, int k) const { return flx() || IB<T>(g).template zd<0, 0, 1>(i, j, k, i - 1, j, k) ? T(0) : (ld(s.U[2], i, j, k) - ld(s.U[2], i - 1, j, k)) * g.idx; }
    __device__ __forceinline__ T dy_u(int i, int j, int k) const { return fly() || IB<T>(g).template zd<1, 0, 0>(i, j, k, i, j - 1, k) ? T(0) : (ld(s.U[0], i, j, k) - ld(s.U[0], i, j - 1, k)) * g.idy; }
    __device__ __forceinline__ T dy_w(int i, int j, int k) const { return fly() || IB<T>(g).template zd<0, 0, 1>(i, j, k, i, j - 1, k) ? T(0) : (ld(s.U[2], i, j, k) - ld(s.U[2], i, j - 1, k)) * g.idy; }
    __device__ __forceinline__ T dz_u(int i, int j, int k) const { return flz() || IB<T>(g).template zd<1, 0, 0>(i, j, k, i, j, k - 1) ? T(0) : (ld(s.U[0], i, j, k) - ld(s.U[0], i, j, k - 1)) * g.idzf[k]; }
    __device__ __forceinline__ T dz_v(int i, int j, int k) const { return flz() || IB<T>(g).template zd<0, 1, 0>(i, j, k, i, j, k - 1) ? T(0) : (ld(s.U[1], i, j, k) - ld(s.U[1], i, j, k - 1)) * g.idzf[k]; }
    __device__ __forceinline__ T dxc(const T *c, int i, int j, int k) const { return flx() || IB<T>(g).template zd<0, 0, 0>(i, j, k, i - 1, j, k) ? T(0) : (ld(c, i, j, k) - ld(c, i - 1, j, k)) * g.idx; }
    __device__ __forceinline__ T dyc(const T *c, int i, int j, int k) const { return fly() || IB<T>(g).template zd<0, 0, 0>(i, j, k, i, j - 1, k) ? T(0) : (ld(c, i, j, k) - ld(c, i, j - 1, k)) * g.idy; }
    __device__ __forceinline__ T dzc(const T *c, int i, int j, int k) const { return flz() || IB<T>(g).template zd<0, 0, 0>(i, j, k, i, j, k - 1) ? T(0) : (ld(c, i, j, k) - ld(c, i, j, k - 1)) * g.idzf[k]; }
    __device__ __forceinline__ T S12(int i, int j, int k) const { return T(0.5) * (dy_u(i, j, k) + dx_v(i, j, k)); }
    __device__ __forceinline__ T S13(int i, int j, int k) const { return T(0.5) * (dz_u(i, j, k) + dx_w(i, j, k)); }
    __device__ __forceinline__ T S23(int i, int j, int k) const { return T(0.5) * (dz_v(i, j, k) + dy_w(i, j, k)); }

    // ================= eddy viscosity at the stress locations (abstract_scalar_diffusivity_closure.jl:343-353)
    __device__ __forceinline__ T nu_ccc(int i, int j, int k) const {
        if (ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) return ph.c0;
        return ld(s.nu, i, j, k);
    }
    __device__ __forceinline__ T nu_ffc(int i, int j, int k) const {
        if (ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) return ph.c0;
        const T *n = s.nu;
        T a = flx() ? ld(n, i, j - 1, k) : T(0.5) * (ld(n, i - 1, j - 1, k) + ld(n, i, j - 1, k));
        T b = flx() ? ld(n, i, j, k) : T(0.5) * (ld(n, i - 1, j, k) + ld(n, i, j, k));
        if (fly()) return b;
        return T(0.5) * (a + b);
    }
    __device__ __forceinline__ T nu_fcf(int i, int j, int k) const {
        if (ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) return ph.c0;
        const T *n = s.nu;
        T a = flx() ? ld(n, i, j, k - 1) : T(0.5) * (ld(n, i - 1, j, k - 1) + ld(n, i, j, k - 1));
        T b = flx() ? ld(n, i, j, k) : T(0.5) * (ld(n, i - 1, j, k) + ld(n, i, j, k));
        if (flz()) return b;
        return T(0.5) * (a + b);
    }
    __device__ __forceinline__ T nu_cff(int i, int j, int k) const {
        if (ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) return ph.c0;
        const T *n = s.nu;
        T a = fly() ? ld(n, i, j, k - 1) : T(0.5) * (ld(n, i, j - 1, k - 1) + ld(n, i, j, k - 1));
        T b = fly() ? ld(n, i, j, k) : T(0.5) * (ld(n, i, j - 1, k) + ld(n, i, j, k));
        if (flz()) return b;
        return T(0.5) * (a + b);
    }
    // tracer diffusivity at fcc / cfc / ccf
    __device__ __forceinline__ T kap_f(int n, int i, int j, int k, int di, int dj, int dk) const {
        if (ph.closure == OM_CLOSURE_SCALAR_DIFFUSIVITY) return ph.c1;
        if (ph.closure == OM_CLOSURE_AMD) return T(0.5) * (ld(s.kap[n], i - di, j - dj, k - dk) + ld(s.kap[n], i, j, k));
        return (T(0.5) * (ld(s.nu, i - di, j - dj, k - dk) + ld(s.nu, i, j, k))) / ph.c2;
    }

    // ∇·U at a cell centre (divergence_operators.jl:16-19), conditional δ on an immersed grid;
    // ip, jp address the i + 1, j + 1 neighbours (wrapped by a caller whose halos are stale)
    __device__ __forceinline__ T divU(int i, int j, int k, int ip, int jp) const {
        const IB<T> ib(g);
        const T *u = s.U[0], *v = s.U[1], *w = s.U[2];
        T sx = flx() || ib.template zd<1, 0, 0>(i, j, k, i + 1, j, k) ? T(0) : Axc(k) * ld(u, ip, j, k) - Axc(k) * ld(u, i, j, k);
        T sy = fly() || ib.template zd<0, 1, 0>(i, j, k, i, j + 1, k) ? T(0) : Ayc(k) * ld(v, i, jp, k) - Ayc(k) * ld(v, i, j, k);
        T sz = flz() || ib.template zd<0, 0, 1>(i, j, k, i, j, k + 1) ? T(0) : g.Az * ld(w, i, j, k + 1) - g.Az * ld(w, i, j, k);
        return iVc(k) * ((sx + sy) + sz);
    }

    // viscous and diffusive fluxes (abstract_scalar_diffusivity_closure.jl:214-262), zero on the
    // immersed periphery of their location (immersed_diffusive_fluxes.jl:25-42)
    __device__ __forceinline__ T f_ux(int i, int j, int k) const { return IB<T>(g).template iper<0, 0, 0>(i, j, k) ? T(0) : T(-2) * (nu_ccc(i, j, k) * dx_u(i, j, k)); }
    __device__ __forceinline__ T f_uy(int i, int j, int k) const { return IB<T>(g).template iper<1, 1, 0>(i, j, k) ? T(0) : T(-2) * (nu_ffc(i, j, k) * S12(i, j, k)); }
    __device__ __forceinline__ T f_uz(int i, int j, int k) const { return IB<T>(g).template iper<1, 0, 1>(i, j, k) ? T(0) : T(-2) * (nu_fcf(i, j, k) * S13(i, j, k)); }
    __device__ __forceinline__ T f_vy(int i, int j, int k) const { return IB<T>(g).template iper<0, 0, 0>(i, j, k) ? T(0) : T(-2) * (nu_ccc(i, j, k) * dy_v(i, j, k)); }
    __device__ __forceinline__ T f_vz(int i, int j, int k) const { return IB<T>(g).template iper<0, 1, 1>(i, j, k) ? T(0) : T(-2) * (nu_cff(i, j, k) * S23(i, j, k)); }
    __device__ __forceinline__ T f_wz(int i, int j, int k) const { return IB<T>(g).template iper<0, 0, 0>(i, j, k) ? T(0) : T(-2) * (nu_ccc(i, j, k) * dz_w(i, j, k)); }
    __device__ __forceinline__ T q_x(int n, const T *c, int i, int j, int k) const { return IB<T>(g).template iper<1, 0, 0>(i, j, k) ? T(0) : -kap_f(n, i, j, k, 1, 0, 0) * dxc(c, i, j, k); }
    __device__ __forceinline__ T q_y(int n, const T *c, int i, int j, int k) const { return IB<T>(g).template iper<0, 1, 0>(i, j, k) ? T(0) : -kap_f(n, i, j, k, 0, 1, 0) * dyc(c, i, j, k); }
    __device__ __forceinline__ T q_z(int n, const T *c, int i, int j, int k) const { return IB<T>(g).template iper<0, 0, 1>(i, j, k) ? T(0) : -kap_f(n, i, j, k, 0, 0, 1) * dzc(c, i, j, k); }

    __device__ __forceinline__ T buoy(int i, int j, int k) const {
        if (ph.buoyancy == OM_BUOYANCY_TRACER) return ld(s.btr, i, j, k);
        if (ph.buoyancy == OM_BUOYANCY_LINEAR_EOS)
            return ph.g * (ph.alpha * ld(s.Ttr, i, j, k) - ph.beta * ld(s.Str, i, j, k));
        return T(0);
    }
    // b(i, j, k) − b(i − di, j − dj, k), formed from the tracers' differences (exact in FP32 for
    // neighbouring values within a factor two of each other, Sterbenz), not from two rounded b
    __device__ __forceinline__ T buoy_diff(int i, int j, int k, int di, int dj) const {
        if (ph.buoyancy == OM_BUOYANCY_TRACER) return ld(s.btr, i, j, k) - ld(s.btr, i - di, j - dj, k);
        if (ph.buoyancy == OM_BUOYANCY_LINEAR_EOS)
            return ph.g * (ph.alpha * (ld(s.Ttr, i, j, k) - ld(s.Ttr, i - di, j - dj, k)) -
                           ph.beta * (ld(s.Str, i, j, k) - ld(s.Str, i - di, j - dj, k)));
        return T(0);
    }
    __device__ __forceinline__ T dzb(int i, int j, int k) const {  // ∂z_b at ccf
        if (ph.buoyancy == OM_BUOYANCY_TRACER) return dzc(s.btr, i, j, k);
        if (ph.buoyancy == OM_BUOYANCY_LINEAR_EOS)
            return ph.g * (ph.alpha * dzc(s.Ttr, i, j, k) - ph.beta * dzc(s.Str, i, j, k));
        return T(0);
    }
};

template <class T> struct HaloJob {
    T *f[kMaxFields + 4];
    int kind_bottom[kMaxFields + 4], kind_top[kMaxFields + 4];   // OM_BC_* ; -1 = w normal flow; -2 = skip
    T val_bottom[kMaxFields + 4], val_top[kMaxFields + 4];
    int nf;
};

// the argument pack of a kernel that takes only the model context
template <class T> struct CtxArgs {
    Ctx<T> C;
};

template <class T> struct RKArgs {
    StepScalar<T> dt;
    T gamma, zeta;
    int first;
    int nfields;
};

// One stage of a mixed-radix line transform of length n (not a power of two): its radix, the
// product m of the radices before it, and ⌈2³²/m⌉, ⌈2³²/(n/radix)⌉.  The high word of t·⌈2³²/d⌉ is
// ⌊t/d⌋ whenever t·(d − 1) < 2³²; here t < 4096 and d ≤ 4096 (R·n ≤ 4096 elements per block);
// the stages treat d = 1 apart.
struct FftStage {
    uint32_t radix, m, mul_m, mul_b;
};
// the stages of a line of length n, ended by radix 0.  The odd radices come first: their stages then
// run at odd sub-lengths, whose output strides spread over the LDS banks.
inline std::vector<FftStage> fft_stages(int n) {
    std::vector<FftStage> st;
    uint32_t m = 1;
    auto mul = [](uint32_t d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
    auto add = [&](uint32_t r) {
        st.push_back(FftStage{r, m, mul(m), mul((uint32_t)n / r)});
        m *= r;
    };
    int rest = n;
    for (int r : {7, 5, 3}) for (; rest % r == 0; rest /= r) add((uint32_t)r);
    int twos = 0;
    for (; rest % 2 == 0; rest /= 2) ++twos;
    for (int r = 11; rest > 1; r += 2) {
        if (r * r > rest) r = rest;
        for (; rest % r == 0; rest /= r) add((uint32_t)r);
    }
    for (; twos >= 2; twos -= 2) add(4);
    if (twos) add(2);
    st.push_back(FftStage{0, 0, 0, 0});
    return st;
}

// Poisson solver plan: spectral storage and per-axis tables (device pointers).
template <class T> struct PoissonPlan {
    typename Vec2<T>::type *S;          // complex spectral array, Ms · Ny · Nz (x rows padded to Ms)
    int Ms;                              // row stride of S: Mx = Nx/2 + 1 rounded up to a 128-byte line
    const typename Vec2<T>::type *tw_xh; // twiddles for the x line (length Nx/2 when Nx is even, Nx otherwise)
    const typename Vec2<T>::type *post;  // exp(-2πi k / Nx), k = 0 .. Nx/2
    const typename Vec2<T>::type *tw_y;  // length Ny
    const typename Vec2<T>::type *tw_z;  // length Nz
    const FftStage *st_x, *st_y, *st_z;  // stages of the x, y and z lines (lengths as the tables')
    const typename Vec2<T>::type *tw_dct; // exp(-iπk / 2Nz), k < Nz (zmode 1)
    const T *lx, *ly, *lz;               // eigenvalues (lz: Nz entries, 2·Nz for Bounded z)
    int zmode;                           // 0 Periodic z, 1 Bounded z via a length-Nz DCT
    int Lz_norm;                         // normalisation of the z transform pair: Nz (Periodic), 2·Nz (Bounded)
    int tridiagonal;                     // Fourier–tridiagonal z solve (stretched z)
};

// Lines of the FFT passes staged per block: the largest power of two R ≤ 16 with R·n ≤ 4096 whose
// R rows (stride n + 1 when R > 1) and `tables` complex table entries fit in 64 KiB of LDS, with a
// second buffer when n is not a power of two (mixed radix).  0: not even one line fits.
inline int fft_lines_per_block(int n, int tables, size_t elem) {
    const bool p2 = (n & (n - 1)) == 0;
    for (int R = 16; R >= 1; R >>= 1) {
        if ((size_t)R * n > 4096) continue;
        const size_t ld = R > 1 ? (size_t)n + 1 : (size_t)n;
        if (((size_t)(p2 ? 1 : 2) * R * ld + (size_t)tables) * elem <= 65536) return R;
    }
    return 0;
}

// table entries of a z line: its twiddles and, with Bounded z, the DCT's c_k
inline int z_line_tables(int Nz, bool bounded) { return bounded ? 2 * Nz : Nz; }

// Levels per block (the z chunk) of a kernel whose blocks march up a tile of columns.  With n =
// tiles · chunks blocks, m = n / CUs of them per CU and `occ` resident at once, a level of a full CU
// costs each block one unit of VALU time, a level of a lone block `lat` units of latency, and a block
// `over` levels beyond its chunk (the state below it; `over_lat` where latency rules).  The last,
// partly filled round of blocks adds up to a lone block's time:
//   cost(chunk) = max((chunk + over) (m + lat (1 − frac q) / max(1, ⌊q⌋)), (chunk + over_lat) lat),  q = m / occ.
// The constants are fits of measured launches of 32³ to 512 × 512 × 256 cells at chunks of 1 to 128
// (tendencies of 32³ FP32: 103 µs at the former fixed chunk of 16, 16 at 1; 128³ 110 → 99;
// 256 × 256 × 128 369 → 350).  Chunks do not change results.
struct MarchCost {
    int occ;
    double lat, over, over_lat;
};
// The chunk for one launch over the given grids (a batch's members share one: a member with longer
// chunks than the rest would end the launch alone).
struct MarchGrid {
    int tiles, Nz;
};
inline int march_chunk(const std::vector<MarchGrid> &grids, int cus, const MarchCost &M) {
    int best = 1, most = 1;
    for (const MarchGrid &g : grids) most = std::max(most, std::min(g.Nz, 64));
    double least = INFINITY, before = 0;
    for (int kc = 1; kc <= most; ++kc) {
        double blocks = 0;
        for (const MarchGrid &g : grids) blocks += (double)g.tiles * ((g.Nz + kc - 1) / kc);
        if (blocks == before) continue;   // the same chunks, less evenly filled
        before = blocks;
        const double m = blocks / cus, q = m / M.occ, f = q - std::floor(q);
        const double tail = f > 0 ? M.lat * (1.0 - f) / std::max(1.0, std::floor(q)) : 0.0;
        const double c = std::max((kc + M.over) * (m + tail), (kc + M.over_lat) * M.lat);
        if (c < 0.999 * least) { least = c; best = kc; }
    }
    return best;
}
inline MarchCost tend_march_cost(size_t elem, int n_tracers) {
    if (elem == 8) return MarchCost{2, 1.4, 0.65, 1.6};
    return n_tracers <= 1 ? MarchCost{5, 2.4, 0.65, 1.6} : MarchCost{4, 2.1, 0.65, 1.6};
}
inline MarchCost centered_march_cost(size_t elem) { return elem == 8 ? MarchCost{4, 2.0, 0.5, 3.0} : MarchCost{6, 2.5, 0.5, 3.0}; }
inline MarchCost closure_march_cost(size_t elem) {
    return elem == 8 ? MarchCost{2, 1.2, 0.35, 2.9} : MarchCost{5, 2.0, 0.8, 2.9};
}
constexpr int kTendTile = 15, kClosureTile = 16;   // cells per tile edge of the two kernels
constexpr int kCenteredX = 32, kCenteredY = 8;     // and of the centered tendency kernel's tile
inline int march_tiles(int Nx, int Ny, int ex, int ey) { return ((Nx + ex - 1) / ex) * ((Ny + ey - 1) / ey); }

// The generic kernels over every cell, or (fixup) only over the cells below kfix of an immersed
// grid, after the tiled kernels have covered the rest
constexpr int kImmersedReach = 5;   // farthest offset of an immersed-boundary query from its cell, plus one
constexpr int kGenericBlockX = 64, kGenericBlockY = 4;   // block shape of k_tendencies / k_closure
// A wave's tile of columns in the fix-up launches.  The cells to redo follow the bottom, so narrow tiles
// fit them better (256 × 256 × 128 seamount: 81 % of the lanes at work; 53 % with the rows of 64 of a
// full launch), and 16 FP32 values are still half a line.
constexpr int kFixX = 16, kFixY = 4;
template <class T> void launch_tendencies(const Ctx<T> &C, hipStream_t st, bool fixup = false);
// z-marching tendency kernels: WENO(order=5) (om_tend_tiled.hip) and Centered(order=2) with constant or
// no diffusivity (om_tend_centered.hip), and the configurations they cover
template <class T> bool centered_tendencies_supported(const Ctx<T> &C);
template <class T> void launch_tend_centered(const Ctx<T> &C, int kchunk, hipStream_t st);
template <class T> bool tiled_tendencies_supported(const Ctx<T> &C);
template <class T> void launch_tend_tiled(const Ctx<T> &C, int kchunk, hipStream_t st);
// Flat z, Periodic x and y, no immersed bottom (om_kernels.hip)
template <class T> bool flat_tendencies_supported(const Ctx<T> &C);
template <class T> void launch_tend_flat(const Ctx<T> &C, hipStream_t st);
template <class T> void launch_closure(const Ctx<T> &C, hipStream_t st, bool fixup = false);
// z-marching LDS-tiled eddy viscosity / diffusivity kernel (om_closure_tiled.hip)
template <class T> bool tiled_closure_supported(const Ctx<T> &C);
template <class T> void launch_closure_tiled(const Ctx<T> &C, int kchunk, hipStream_t st);
template <class T> void launch_hydrostatic(const Ctx<T> &C, hipStream_t st);
template <class T> void launch_rk3(const Ctx<T> &C, StepScalar<T> dt, T gamma, T zeta, int first, int nfields, hipStream_t st);
// U −= dtp·∇p (phi = 0: p is the pressure) or U −= ∇ϕ (phi = 1: ϕ = p·Δt, as the reference stores it)
// wrap = 1: periodic x and y without an immersed bottom; p's halos are not read
template <class T> void launch_correct(const Ctx<T> &C, StepScalar<T> dtp, int phi, hipStream_t st, int wrap = 0);
// mask_immersed_field! of a field at location loc (0 ccc, 1 fcc, 2 cfc, 3 ccf) on an immersed grid
// (launch_mask_velocities: u, v and w at theirs)
template <class T> void launch_mask(const DevGrid<T> &g, T *f, int loc, hipStream_t st);
template <class T> void launch_mask_velocities(const DevGrid<T> &g, T *const *U, hipStream_t st);
// conjugate-gradient Poisson solver kernels (om_cg.hip)
// Grid-wide reductions of the elementwise kernels use kCgRedBlocks blocks (and partial sums per
// value).  The 7-point operator sweeps take a 64 × 4 tile of columns and a chunk of kchunk levels
// per block, with the chunk length chosen so that the grid holds at most kCgStencilPartials blocks
// where the tiles allow it; cg_partials_needed is the partial-sum buffer a solver allocates.
constexpr int kCgRedBlocks = 2048;
constexpr int kCgStTx = 64, kCgStTy = 4;
constexpr int kCgStencilPartials = 4096;
constexpr int kCgStBatch = 4;      // levels per batch of loads in a sweep
constexpr int kCgStMinChunk = 32;  // levels per thread where the grid allows it
struct CgStencilShape {
    int ntx, nty, kchunk, nblocks;
};
inline CgStencilShape cg_stencil_shape(int Nx, int Ny, int Nz) {
    CgStencilShape s;
    s.ntx = (Nx + kCgStTx - 1) / kCgStTx;
    s.nty = (Ny + kCgStTy - 1) / kCgStTy;
    const int tiles = s.ntx * s.nty;
    int nch = std::max(1, std::min((Nz + kCgStMinChunk - 1) / kCgStMinChunk, kCgStencilPartials / tiles));
    s.kchunk = (Nz + nch - 1) / nch;
    nch = (Nz + s.kchunk - 1) / s.kchunk;
    s.nblocks = tiles * nch;
    return s;
}
// The direction sweep's tile and chunk: about kCgDirBlocks blocks (two per CU, all resident at once: 160 VGPRs
// allow three) where the grid allows chunks of eight levels or more (a chunk reads two levels beyond its own).
constexpr int kCgDirX = 64, kCgDirY = 8, kCgDirBlocks = 512;
inline CgStencilShape cg_direction_shape(int Nx, int Ny, int Nz) {
    CgStencilShape s;
    s.ntx = (Nx + kCgDirX - 1) / kCgDirX;
    s.nty = (Ny + kCgDirY - 1) / kCgDirY;
    const int tiles = s.ntx * s.nty;
    int nch = std::max(1, std::min((Nz + 7) / 8, kCgDirBlocks / tiles));
    s.kchunk = (Nz + nch - 1) / nch;
    nch = (Nz + s.kchunk - 1) / s.kchunk;
    s.nblocks = tiles * nch;
    return s;
}
// One of a solver's three sets of partial sums: the sweep that reads one set writes another.
inline size_t cg_partials_needed(int Nx, int Ny, int Nz) {
    return (size_t)std::max(4 * kCgRedBlocks, std::max(cg_stencil_shape(Nx, Ny, Nz).nblocks, 3 * cg_direction_shape(Nx, Ny, Nz).nblocks));
}
// The iteration's scalars stay on the device, in the solver's reduction-output array: slots 0-3
// hold results the host reads; ρ of iteration k sits at
// cg_slot_rho(k) by the parity of k, so that ρ_prev is still there; then the gauge sweep's ‖V⁻¹r‖²
// with the sums of x and r.  The sweeps form α, β and the gauge means from them and from the partial
// sums of the launch before.
constexpr int kCgSlotRho = 8, kCgSlotGauge = 16, kCgSlots = 24;   // Gauge: ‖V⁻¹r‖², Σx, Σr
__host__ __device__ inline int cg_slot_rho(int it) { return kCgSlotRho + 2 * (it & 1); }
template <class T> void cg_scale(const DevGrid<T> &g, T *f, T s, int mode, hipStream_t st);
template <class T> void cg_gather(const DevGrid<T> &g, const double *x, T *dense, hipStream_t st);
template <class T> void cg_xio(const DevGrid<T> &g, T *f, double *x, T s, int store, hipStream_t st);
template <class T> void cg_source(const Ctx<T> &C, const T *dense_rhs, double *b, hipStream_t st);
template <class T> void cg_residual(const DevGrid<T> &g, const double *x, const double *b, double *r, double *partial,
                                    double *out, hipStream_t st);
template <class T> void cg_halo_r(const DevGrid<T> &g, double *r, hipStream_t st);
template <class T> void cg_dd(const DevGrid<T> &g, const double *r, T *z, hipStream_t st);
template <class T> void cg_copy_r(const DevGrid<T> &g, const double *r, T *z, hipStream_t st);
// learned correction to the FFT preconditioner and flexible CG (om_cg.hip)
template <class T> void ln_scales(const DevGrid<T> &g, const double *r, const T *z, double *partial, double *out, hipStream_t st);
template <class T> void ln_input(const DevGrid<T> &g, const double *r, const T *z, double isr, double isz, float *in3, hipStream_t st);
template <class T> void ln_x0(const DevGrid<T> &g, const double *r, const T *z, double isr, double isz, void *x0, hipStream_t st);
template <class T> void ln_correct(const DevGrid<T> &g, T *z, const float *out, double sz, hipStream_t st);
template <class T> void cg_copy_d(const DevGrid<T> &g, const double *src, double *dst, hipStream_t st);
template <class T> void cg_dot2(const DevGrid<T> &g, const T *z, const double *r, const double *rp, double *partial,
                                hipStream_t st);
template <class T> void ln_target(const DevGrid<T> &g, const double *xf, const double *xk, const float *in3k, double isz, float *tgt,
                                  double *partial, double *out, hipStream_t st);
template <class T> void ln_center(const DevGrid<T> &g, float *tgt, float mean, hipStream_t st);
template <class T> void ln_mask(const DevGrid<T> &g, float *mask, hipStream_t st);
// A-energy loss dᵀ(−V∇²)d of d = act·(y − t) (y may be null: d = −t) and, when gout is given,
// gout = −2·gscale·act·V∇²d; dscratch is a padded FP64 field
template <class T> void ln_energy(const DevGrid<T> &g, const float *y, const float *tgt, double *dscratch, double gscale, float *gout,
                                  double *partial, double *out, hipStream_t st);
// ColumnwiseTridiagonalPreconditioner: z = Lz⁻¹ r per column; t is an Nx·Ny·Nz scratch array
template <class T> void cg_ct(const DevGrid<T> &g, const double *r, T *z, T *t, hipStream_t st);
template <class T> void cg_dot_zr(const DevGrid<T> &g, const T *z, const double *r, double *partial, hipStream_t st);
// p = z (first) or z + β p_old, q = V∇²p, with ρ from the dot's partial sums; partial sums of p·q, Σp, Σq (p
// and p_old, dots and partial: different buffers)
template <class T> void cg_direction(const DevGrid<T> &g, const T *z, const double *pold, double *p, double *q, const double *dots,
                                     double *sc, int it, int first, int flex, double *partial, hipStream_t st);
// The gauge and norm sweep (step = 0: the solve's first; step = 1: with the iteration's update of
// x and r folded in, from the direction sweep's partial sums pq); writes ‖V⁻¹r‖², Σx, Σr to out and the
// first to host memory too.  dense: also write r V⁻¹ in FP32 cell order,
// the FFT preconditioner's source (may be null).
template <class T> void cg_gauge_norm(const DevGrid<T> &g, double *x, const double *p, double *r, const double *q,
                                      const double *sc, const double *pq, int it, int step, double ncell, T *dense, double *partial,
                                      double *out, double *host, hipStream_t st);
template <class T> void cg_true_residual(const DevGrid<T> &g, const double *x, const double *b, double *e, double *partial,
                                         double *out, hipStream_t st);
template <class T> void cg_gauged_norm(const DevGrid<T> &g, const double *e, double mean, double *partial, double *out,
                                       hipStream_t st);
template <class T> void launch_divergence(const Ctx<T> &C, T *out, hipStream_t st);
// mem[0 .. 3] ← v: the numbers of a captured step (StepScalar)
template <class T> struct StepTimes {
    T v[4];
};
template <class T> void launch_step_times(const StepTimes<T> &t, T *mem, hipStream_t st);
template <class T> void launch_halos(const DevGrid<T> &g, const HaloJob<T> &J, hipStream_t st);
// whether the X-forward pass forms ∇·U of the state without reading a halo
template <class T> bool poisson_source_reads_no_halo(const Ctx<T> &C) {
    return !C.g.kbot && C.g.tx != OM_FLAT && C.g.ty != OM_FLAT;
}
// Solve ∇²ϕ = source; writes ϕ / divisor into `out` (the nonhydrostatic pressure p/Δt when
// called from the pressure correction, divisor = 1 otherwise).
template <class T> void launch_poisson(const PoissonPlan<T> &P, const Ctx<T> &C, const T *src, T *out, int dense_out,
                                       StepScalar<T> divisor, hipStream_t st);

// FP64 iterative refinement of a Poisson solve.  Residual r = b − ∇²p in FP64 arithmetic, stored
// dense in T: ∇² is the operator the FFT / Fourier–tridiagonal solver inverts (periodic x, y;
// Neumann walls on a Bounded z; ihx2 etc. the FP64 inverse squared spacings of its eigenvalues),
// evaluated without halos; p has element strides psy, psz.  b: b64 (dense FP64) if given, else the
// FP64 divergence of the velocities of C divided by `divisor`.  Then p += d (dense correction).
struct RefineOp {
    double ihx2, ihy2, ihz2;   // ihz2 < 0: stretched z, coefficients from idzf, idzc
    const double *idzf;        // FP64 1/Δzᶠ at faces k = 0 .. Nz and 1/Δzᶜ of cells k = 0 .. Nz − 1,
    const double *idzc;        // from the configuration's FP64 face heights (stretched z)
};
template <class T> void launch_poisson_residual(const Ctx<T> &C, const RefineOp &L, const T *p, int64_t psy, int64_t psz,
                                                const double *b64, StepScalar<T> divisor, T *r, hipStream_t st);
template <class T> void launch_add_correction(const DevGrid<T> &g, T *p, int64_t psy, int64_t psz, const T *d, hipStream_t st);

// diagnostics reductions (om_diagnostics.hip); partial holds 3·1024 doubles, out 3 doubles
// (max, min, NaN count); the advection timescale reduction leaves max = max inverse timescale
template <class T> void launch_adv_timescale(const Ctx<T> &C, double *partial, double *out, hipStream_t st);
// allocation-free reductions: the device address of the library's static scratch array on `device`
// (taken once per device; nullptr with *err set on failure), its size and the part the partials take
double *diag_scratch(int device, int *err);
int diag_scratch_doubles();
int diag_partial_doubles();
constexpr int64_t kNoallocMaxElements = int64_t(1) << 40;
template <class T> void launch_field_stats(const DevGrid<T> &g, const T *origin, int with_halos, int face_z, double *partial,
                                           double *out, hipStream_t st);

}  // namespace om
