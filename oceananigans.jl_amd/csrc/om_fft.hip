// om_fft.hip — pressure Poisson solvers on gfx950.
//
// Spectral array S (complex, x fastest): S[(k·Ny + j)·Ms + kx], kx < Mx = Nx/2 + 1 (real-to-complex
// along a Periodic x) or 1 (Flat x); the row stride Ms rounds Mx up to a 128-byte line, and the
// passes skip the padding entries kx ≥ Mx.  Passes, each one HBM read + one write of S:
//   X-forward  : source term (∇·U* formed on the fly, optionally ×Δzᶜ) → real-to-complex FFT
//   Y-forward  : complex FFT along y                    (skipped when y is the last axis)
//   last axis  : forward transform · eigenvalue division · backward transform in one kernel
//                (Bounded z: DCT-II / DCT-III pair through one complex FFT of length Nz;
//                 Fourier–tridiagonal: Thomas algorithm)
//   Y-backward, X-backward (complex-to-real, written into the pressure field's interior)
// Each line transform is an in-place radix-4 Stockham FFT in LDS for power-of-two lengths and a
// mixed-radix Stockham FFT between two LDS buffers otherwise; the global loads that stage the lines are batched per thread.  Reference: src/Solvers/fft_based_poisson_solver.jl:94-124,
// src/Solvers/fourier_tridiagonal_poisson_solver.jl:231-260, src/Solvers/batched_tridiagonal_solver.jl:211-243.
#include <hip/hip_runtime.h>

#include <limits>
#include <stdexcept>

#include "om_internal.h"
#include "om_batch.h"
#include "om_kernels.h"

namespace om {

template <class T> using C2 = typename Vec2<T>::type;

template <class T> __device__ __forceinline__ C2<T> cadd(C2<T> a, C2<T> b) { C2<T> r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
template <class T> __device__ __forceinline__ C2<T> csub(C2<T> a, C2<T> b) { C2<T> r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }
template <class T> __device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b) { C2<T> r; r.x = a.x * b.x - a.y * b.y; r.y = a.x * b.y + a.y * b.x; return r; }
template <class T> __device__ __forceinline__ C2<T> cconj(C2<T> a) { a.y = -a.y; return a; }
template <class T> __device__ __forceinline__ C2<T> cmk(T x, T y) { C2<T> r; r.x = x; r.y = y; return r; }

// Global → LDS staging.  get(t) issues the global loads of element t, put(t, v) stores it in LDS.
// Each thread first issues the loads of B elements and only then stores them, so a wave keeps B
// loads in flight (a plain load-then-store loop waits out the full memory latency per element).
template <int B, class Get, class Put>
__device__ __forceinline__ void staged_copy(int count, Get get, Put put) {
    const int nt = blockDim.x;
    for (int t0 = threadIdx.x; t0 < count; t0 += B * nt) {
        decltype(get(0)) v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int t = t0 + u * nt;
            if (t < count) v[u] = get(t);
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int t = t0 + u * nt;
            if (t < count) put(t, v[u]);
        }
    }
}

// Butterfly of P points, P odd: y_q = Σ_p c_p e^{∓2πi pq/P}, from the sums and differences of the
// pairs (c_k, c_{P−k}): y_q, y_{P−q} = A ∓ iB (forward) with A = c_0 + Σ_k cos(2πkq/P) (c_k + c_{P−k}) and
// B = Σ_k sin(2πkq/P) (c_k − c_{P−k}).  cs, sn: cos and sin of 2πm/P, m = 0 .. P−1.
template <int P> struct OddTable;
template <> struct OddTable<3> {
    static constexpr double cs[3] = {1.0, -0.5, -0.5};
    static constexpr double sn[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
};
template <> struct OddTable<5> {
    static constexpr double cs[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410, 0.30901699437494742410};
    static constexpr double sn[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917, -0.95105651629515357212};
};
template <> struct OddTable<7> {
    static constexpr double cs[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                                     -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
    static constexpr double sn[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048,
                                     -0.43388373911755812048, -0.97492791218182360702, -0.78183148246802980871};
};
template <class T, int P> __device__ __forceinline__ void butterfly(C2<T> (&c)[P], bool inverse) {
    if constexpr (P == 2) {
        const C2<T> t = csub<T>(c[0], c[1]);
        c[0] = cadd<T>(c[0], c[1]);
        c[1] = t;
    } else if constexpr (P == 4) {
        const C2<T> t0 = cadd<T>(c[0], c[2]), t1 = csub<T>(c[0], c[2]), t2 = cadd<T>(c[1], c[3]), d = csub<T>(c[1], c[3]);
        const C2<T> t3 = inverse ? cmk<T>(-d.y, d.x) : cmk<T>(d.y, -d.x);   // ±i·(c1 − c3)
        c[0] = cadd<T>(t0, t2);
        c[1] = cadd<T>(t1, t3);
        c[2] = csub<T>(t0, t2);
        c[3] = csub<T>(t1, t3);
    } else {
        constexpr int H = (P - 1) / 2;
        C2<T> sp[H], dm[H];
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            sp[k - 1] = cadd<T>(c[k], c[P - k]);
            dm[k - 1] = csub<T>(c[k], c[P - k]);
        }
        const C2<T> c0 = c[0];
#pragma unroll
        for (int k = 0; k < H; ++k) c[0] = cadd<T>(c[0], sp[k]);
#pragma unroll
        for (int q = 1; q <= H; ++q) {
            C2<T> A = c0, B = cmk<T>(T(0), T(0));
#pragma unroll
            for (int k = 1; k <= H; ++k) {
                const T cs = T(OddTable<P>::cs[k * q % P]), sn = T(OddTable<P>::sn[k * q % P]);
                A.x += cs * sp[k - 1].x;
                A.y += cs * sp[k - 1].y;
                B.x += sn * dm[k - 1].x;
                B.y += sn * dm[k - 1].y;
            }
            if (inverse) B = cmk<T>(-B.x, -B.y);
            c[q] = cmk<T>(A.x + B.y, A.y - B.x);       // A − iB
            c[P - q] = cmk<T>(A.x - B.y, A.y + B.x);   // A + iB
        }
    }
}

// One Stockham stage of radix P on R lines of length n, a → b: at sub-length m the butterfly
// bf = kk + jj·m (kk < m) of a line takes a[bf + p·n/P] to b[kk + (jj·P + q)·m], times w^{q·jj·m}.
// The butterflies of all lines are one flat range; bf and jj come from multiplications by the
// stage's reciprocals (exact for the ranges here, see FftStage).
template <class T, int P>
__device__ __forceinline__ void fft_stage(const C2<T> *a, C2<T> *b, int R, int n, int ld, const C2<T> *tw, bool inverse,
                                          const FftStage &S) {
    const int nb = n / P, m = (int)S.m;
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));   // keeps each radix's index arithmetic inside its own case
#pragma unroll 1
    for (; t < R * nb; t += blockDim.x) {
        const int row = nb == 1 ? t : (int)__umulhi((uint32_t)t, S.mul_b), bf = t - row * nb;
        const int jj = m == 1 ? bf : (int)__umulhi((uint32_t)bf, S.mul_m), kk = bf - jj * m;
        const C2<T> *src = a + row * ld + bf;
        C2<T> c[P];
#pragma unroll
        for (int p = 0; p < P; ++p) c[p] = src[p * nb];
        butterfly<T, P>(c, inverse);
        C2<T> *dst = b + row * ld + kk + jj * P * m;
        const int e = jj * m;
        dst[0] = c[0];
#pragma unroll
        for (int q = 1; q < P; ++q) {
            C2<T> w = tw[q * e];
            if (inverse) w.y = -w.y;
            dst[q * m] = cmul<T>(w, c[q]);
        }
    }
}

// The same stage for any radix: one output per thread, a direct sum over the P inputs.
template <class T>
__device__ __forceinline__ void fft_stage_any(const C2<T> *a, C2<T> *b, int R, int n, int ld, const C2<T> *tw, bool inverse,
                                              const FftStage &S) {
    const int P = (int)S.radix, nb = n / P, m = (int)S.m;
#pragma unroll 1
    for (int t = threadIdx.x; t < R * n; t += blockDim.x) {
        const int row = t / n, o = t - row * n;
        const int v = o / m, kk = o - v * m, jj = v / P, q = v - jj * P;
        const C2<T> *src = a + row * ld + kk + jj * m;
        C2<T> s = src[0];
        int f = 0;
#pragma unroll 2
        for (int p = 1; p < P; ++p) {
            f += q;
            if (f >= P) f -= P;
            C2<T> w = tw[f * nb];
            if (inverse) w.y = -w.y;
            s = cadd<T>(s, cmul<T>(src[p * nb], w));
        }
        C2<T> w = tw[q * jj * m];
        if (inverse) w.y = -w.y;
        b[row * ld + o] = cmul<T>(w, s);
    }
}

// R lines of length n, row r at a + r·ld; tw (in LDS) holds exp(-2πi m / n), m < n.  Returns the
// buffer that holds the (unnormalised) transform.
// MIXED = false, power-of-two n: in-place Stockham stages of radix 4 (one radix-2 stage first when
// log2 n is odd).  A radix-R stage at sub-length m maps a[kk + jj·m + p·n/R] (p < R) to
// a[kk + R·jj·m + q·m] = w^{q·jj·m} Σ_p c_p e^{∓2πi pq/R}; every thread reads its butterflies'
// inputs into registers, the block synchronises, and the outputs overwrite the same buffer, so
// one buffer serves every stage.  Each thread holds at most 2 radix-4 (4 radix-2) butterflies:
// R·n ≤ 8·blockDim.x.  Index splits are shifts and masks.
// MIXED = true, other n: the stages of the plan (radices 7, 5, 3, then any prime above 7 as a direct
// sum of that length, then 4 and 2), each from one buffer to the other.  LDS traffic and barriers
// bound it (an FP32 y pass of 192 × 192 × 96 takes 14 µs, 3.9 TB/s, against 318 µs as direct sums of
// 192 terms; the z pass of 150 × 100 × 75 12 µs against 284 as a 150-point even extension).
// The two are separate kernels: in one, the radix-7 butterfly's registers would halve the blocks a
// CU holds of the power-of-two passes too (98 VGPRs against 54).
template <class T, bool MIXED>
__device__ __forceinline__ C2<T> *lds_fft(C2<T> *a, C2<T> *b, int R, int n, int ld, const C2<T> *tw, bool inverse,
                       const FftStage *__restrict__ stages) {
    const int nt = blockDim.x;
    const int tid = threadIdx.x;
    if constexpr (!MIXED) {
        const int lg = __builtin_ctz((unsigned)n);
        int lm = 0;   // log2 of the current sub-length m
        if (lg & 1) {
            const int half = n >> 1, lh = lg - 1, nb = R * half;
            C2<T> c0[4], c1[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = tid + u * nt;
                if (t < nb) {
                    const int base = (t >> lh) * ld + (t & (half - 1));
                    c0[u] = a[base];
                    c1[u] = a[base + half];
                }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = tid + u * nt;
                if (t < nb) {
                    const int jj = t & (half - 1);
                    C2<T> w = tw[jj];
                    if (inverse) w.y = -w.y;
                    const int ob = (t >> lh) * ld + (jj << 1);
                    a[ob] = cadd<T>(c0[u], c1[u]);
                    a[ob + 1] = cmul<T>(w, csub<T>(c0[u], c1[u]));
                }
            }
            __syncthreads();
            lm = 1;
        }
        const int quarter = n >> 2, lq = lg - 2, nb = R * quarter;
        for (; lm < lg; lm += 2) {
            const int m = 1 << lm;
            C2<T> c[2][4];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = tid + u * nt;
                if (t < nb) {
                    const int ib = (t >> lq) * ld + (t & (quarter - 1));   // = row + kk + jj·m
#pragma unroll
                    for (int p = 0; p < 4; ++p) c[u][p] = a[ib + p * quarter];
                }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = tid + u * nt;
                if (t < nb) {
                    const int bf = t & (quarter - 1);
                    const int jj = bf >> lm, kk = bf & (m - 1);
                    const C2<T> t0 = cadd<T>(c[u][0], c[u][2]), t1 = csub<T>(c[u][0], c[u][2]);
                    const C2<T> t2 = cadd<T>(c[u][1], c[u][3]), d = csub<T>(c[u][1], c[u][3]);
                    const C2<T> t3 = inverse ? cmk<T>(-d.y, d.x) : cmk<T>(d.y, -d.x);   // ±i·(c1 − c3)
                    const int e = jj << lm;
                    C2<T> w1 = tw[e], w2 = tw[2 * e], w3 = tw[3 * e];
                    if (inverse) { w1.y = -w1.y; w2.y = -w2.y; w3.y = -w3.y; }
                    const int ob = (t >> lq) * ld + kk + (jj << (lm + 2));
                    a[ob] = cadd<T>(t0, t2);
                    a[ob + m] = cmul<T>(w1, cadd<T>(t1, t3));
                    a[ob + 2 * m] = cmul<T>(w2, csub<T>(t0, t2));
                    a[ob + 3 * m] = cmul<T>(w3, csub<T>(t1, t3));
                }
            }
            __syncthreads();
        }
        return a;
    } else {
#pragma unroll 1
        for (int q = 0;; ++q) {
            const FftStage S = stages[q];
            switch (S.radix) {
                case 0: return a;
                case 2: fft_stage<T, 2>(a, b, R, n, ld, tw, inverse, S); break;
                case 3: fft_stage<T, 3>(a, b, R, n, ld, tw, inverse, S); break;
                case 4: fft_stage<T, 4>(a, b, R, n, ld, tw, inverse, S); break;
                case 5: fft_stage<T, 5>(a, b, R, n, ld, tw, inverse, S); break;
                case 7: fft_stage<T, 7>(a, b, R, n, ld, tw, inverse, S); break;
                default: fft_stage_any<T>(a, b, R, n, ld, tw, inverse, S);
            }
            __syncthreads();
            C2<T> *t = a;
            a = b;
            b = t;
        }
    }
}

template <class T> __device__ __forceinline__ void load_table(C2<T> *dst, const C2<T> *src, int n) {
    staged_copy<4>(n, [&](int t) { return src[t]; }, [&](int t, C2<T> v) { dst[t] = v; });
}

constexpr int kXFwdBatch = 4;      // elements per thread and batch of loads of the X-forward source
constexpr int kFftThreads = 512;   // threads per block of the line kernels (a multiple of R ≤ 16)

// Line staging geometry, chosen on the host: R lines per block, row stride ld (n + 1 when R > 1,
// so the R rows start in different LDS banks), tables first, then buffer a, then b (only for a
// length that is not a power of two).
struct LineGeom {
    int R, lgR, ld;
};

// ---------------------------------------------------------------------------------------------
// X-forward: source term → R2C along x.  One block handles R rows (j, k).
// src == nullptr: the source is ∇·U of the state (solve_for_pressure.jl:12-18); else a dense
// interior array.  scale_dzc: multiply by Δzᶜ(k) (Fourier–tridiagonal source, :36-42).
// ---------------------------------------------------------------------------------------------
template <class T> struct XFwdArgs {
    Ctx<T> C;
    const T *src;
    C2<T> *S;
    const C2<T> *tw;      // length Nx/2 table (for the half-length complex FFT), Nx when Nx is odd
    const FftStage *stages;   // of the line length of tw
    const C2<T> *post;    // exp(-2πi k / Nx), k = 0 .. Nx/2
    int scale_dzc;
    // FP32: form the cancelling sum of the divergence with its rounding errors (cancelling_sum).  The
    // velocity differences of a nearly divergence-free flow cancel to a small part of each;
    // rounded term by term they leave white noise of ε|U|/Δx, which the inverse Laplacian amplifies
    // at the longest waves: most of the FP32 pressure's error (1.1e-5 against 2e-6 of FP64 at
    // 192 × 192 × 96 stretched).  On for grids with a line that is not a power of two.  The radix has no part in
    // this: the sum would be better everywhere (a step's largest relative error of u, v, w, b, p at 256 × 256 × 128 3.1e-6 → 1.2e-6,
    // at 512 × 512 × 256 4.5e-5 → 3.1e-5, for 0.2 to 0.4 % of its time), but a pressure moved by the error of the
    // plain sum (4.7e-5 there) is further from earlier results than the better sum brings it to the exact
    // one.  So grids of powers of two keep the plain sum, and their results bit for bit.
    int compensated;
    LineGeom L;
    FastDiv fNy, fMx;
    int Ms;
};

template <class T> __device__ __forceinline__ T source_at(const Ctx<T> &C, int i, int j, int k) {
    // divergence with periodic index wrap in x and y (halos of U* are not needed)
    const int ip = (i + 1 == C.g.Nx) ? 0 : i + 1;
    const int jp = (j + 1 == C.g.Ny) ? 0 : j + 1;
    if (C.g.kbot) return C.divU(i, j, k, ip, jp);
    // without an immersed bottom: Ctx::divU's expression, the six loads addressed from one index
    const int64_t o = C.at(i, j, k);
    const T *u = C.s.U[0] + o, *v = C.s.U[1] + o, *w = C.s.U[2] + o;
    const T sx = C.flx() ? T(0) : C.Axc(k) * u[ip - i] - C.Axc(k) * u[0];
    const T sy = C.fly() ? T(0) : C.Ayc(k) * v[(int64_t)(jp - j) * C.g.sy] - C.Ayc(k) * v[0];
    const T sz = C.flz() ? T(0) : C.g.Az * w[C.g.sz] - C.g.Az * w[0];
    return C.iVc(k) * ((sx + sy) + sz);
}

// A₁(a₁ − b₁) + A₂(a₂ − b₂) + A₃(a₃ − b₃) rounded (nearly) once: each difference and product with its
// rounding error (Knuth's two-sum; the product's by FMA), the errors summed beside the values.
__device__ __forceinline__ float cancelling_sum(float A1, float a1, float b1, float A2, float a2, float b2, float A3, float a3, float b3) {
    auto two_sum = [](float x, float y, float &err) {
        const float s = x + y, yy = s - x;
        err += (x - (s - yy)) + (y - yy);
        return s;
    };
    float err = 0.0f;
    auto term = [&](float A, float a, float b) {
        float e = 0.0f;
        const float d = two_sum(a, -b, e), t = A * d;
        err += fmaf(A, e, fmaf(A, d, -t));
        return t;
    };
    const float t1 = term(A1, a1, b1), t2 = term(A2, a2, b2), t3 = term(A3, a3, b3);
    const float s12 = two_sum(t1, t2, err), s = two_sum(s12, t3, err);
    return s + err;
}
__device__ __forceinline__ double cancelling_sum(double, double, double, double, double, double, double, double, double) { return 0.0; }

// SRC: where the source comes from.  kSrcVelocity: ∇·U without an immersed bottom, read without halos
// (poisson_source_reads_no_halo); kSrcDense: the dense array; kSrcGeneral: ∇·U with every topology
// and bottom test per element.  Variants of one kernel, since the general source alone is
// thousands of instructions that the others would carry.
enum { kSrcGeneral = 0, kSrcVelocity = 1, kSrcDense = 2 };
template <class T, bool MIXED, int SRC> struct KXFwd {
    using Family = KXFwd<T, false, kSrcGeneral>;
    static constexpr int kThreads = kFftThreads, kMinBlocks = 1;
    static __device__ __forceinline__ void run(const XFwdArgs<T> &A, const Blk &B);
};
template <class T, bool MIXED, int SRC> __device__ __forceinline__ void KXFwd<T, MIXED, SRC>::run(const XFwdArgs<T> &A, const Blk &B) {
    extern __shared__ unsigned char smem_raw[];
    const Ctx<T> &C = A.C;
    const int Nx = C.g.Nx, Ny = C.g.Ny;
    const bool half = (Nx & 1) == 0;
    const int M = half ? Nx / 2 : Nx;      // line length of the complex FFT
    const int Mx = Nx / 2 + 1;
    const int R = A.L.R, ld = A.L.ld;
    C2<T> *twl = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *a = twl + M;
    C2<T> *b = a + R * ld;
    const int row0 = B.x * R;
    const int nrows = Ny * C.g.Nz;
    load_table<T>(twl, A.tw, M);
    T *ap = reinterpret_cast<T *>(a);
    // blockDim.x / R threads per row: a thread's row (j, k), its metric factors and addresses are
    // fixed, and its elements i = l, l + tpr, … differ by constant offsets.  Rows past the last stage
    // zeros.
    const int lgt = __builtin_ctz((unsigned)blockDim.x) - A.L.lgR;   // log2 of threads per row
    const int tpr = 1 << lgt;
    const int r = threadIdx.x >> lgt, l = threadIdx.x & (tpr - 1);
    const int row = row0 + r;
    const bool live = row < nrows;
    const int k = live ? (int)fdiv((uint32_t)row, A.fNy) : 0, j = live ? row - k * Ny : 0;
    const T zs = A.scale_dzc && live ? C.g.dzc[k] : T(1);
    auto put = [&](int i, T x) {
        if (half) ap[2 * (r * ld + (i >> 1)) + (i & 1)] = x;
        else a[r * ld + i] = cmk<T>(x, T(0));
    };
    if constexpr (SRC == kSrcVelocity) {
        // each thread forms kXFwdBatch elements at a time from loads all issued before any arithmetic,
        // with no per-element branch.  Its neighbours across periodic edges are read by wrapped
        // index, and a Bounded z's boundary faces of w as the zero the impenetrable fill writes
        // there, so it reads no halo.
        const int jp = (j + 1 == Ny) ? 0 : j + 1;
        const int64_t o = C.at(0, j, k);
        const T *u = C.s.U[0] + o, *v = C.s.U[1] + o, *w = C.s.U[2] + o;
        const bool flat = C.flz();   // (w's differences are zero then)
        const int kp = flat || (C.g.tz == OM_PERIODIC && k + 1 == C.g.Nz) ? 0 : k + 1;
        const T *vp = C.s.U[1] + C.at(0, jp, k), *wp = C.s.U[2] + C.at(0, j, kp);
        const bool wb = C.g.tz == OM_BOUNDED && k == 0, wt = C.g.tz == OM_BOUNDED && k == C.g.Nz - 1;
        const T Ax = C.Axc(k), Ay = C.Ayc(k), Az = C.g.Az, iV = C.iVc(k);
        for (int i0 = l; i0 < Nx; i0 += kXFwdBatch * tpr) {
            T su[kXFwdBatch], sq[kXFwdBatch], sv[kXFwdBatch], svp[kXFwdBatch], sw[kXFwdBatch], swp[kXFwdBatch];
#pragma unroll
            for (int e = 0; e < kXFwdBatch; ++e) {
                const int i = i0 + e * tpr;
                const bool in = live && i < Nx;
                const int ii = in ? i : 0;
                const int ip = (ii + 1 == Nx) ? 0 : ii + 1;
                su[e] = in ? u[ii] : T(0);
                sq[e] = in ? u[ip] : T(0);
                sv[e] = in ? v[ii] : T(0);
                svp[e] = in ? vp[ii] : T(0);
                sw[e] = in && !wb ? w[ii] : T(0);
                swp[e] = in && !wt ? wp[ii] : T(0);
            }
#pragma unroll
            for (int e = 0; e < kXFwdBatch; ++e) {
                const int i = i0 + e * tpr;
                if (i < Nx) {
                    T d;
                    if (sizeof(T) == 4 && A.compensated) {
                        d = iV * cancelling_sum(Ax, sq[e], su[e], Ay, svp[e], sv[e], Az, swp[e], sw[e]);
                    } else {
                        // Ctx::divU's expression (source_at), in its order of operations
                        const T sx = Ax * sq[e] - Ax * su[e];
                        const T sy = Ay * svp[e] - Ay * sv[e];
                        const T sz = flat ? T(0) : Az * swp[e] - Az * sw[e];
                        d = iV * ((sx + sy) + sz);
                    }
                    put(i, A.scale_dzc ? zs * d : d);
                }
            }
        }
    } else {
        constexpr int NB = SRC == kSrcDense ? kXFwdBatch : 4;
        const T *dense = A.src + (int64_t)Nx * (live ? row : 0);
        for (int i0 = l; i0 < Nx; i0 += NB * tpr) {
            T x[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int i = i0 + u * tpr;
                x[u] = T(0);
                if (live && i < Nx) {
                    x[u] = SRC == kSrcDense ? dense[i] : source_at<T>(C, i, j, k);
                    if (A.scale_dzc) x[u] = zs * x[u];
                }
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int i = i0 + u * tpr;
                if (i < Nx) put(i, x[u]);
            }
        }
    }
    __syncthreads();
    const C2<T> *Z = lds_fft<T, MIXED>(a, b, R, M, ld, twl, false, A.stages);
    for (int t = threadIdx.x; t < R * Mx; t += blockDim.x) {
        const int r = (int)fdiv((uint32_t)t, A.fMx), kk = t - r * Mx;
        const int row = row0 + r;
        if (row >= nrows) continue;
        if (!half) { A.S[(int64_t)row * A.Ms + kk] = Z[r * ld + kk]; continue; }
        const C2<T> zk = Z[r * ld + (kk == M ? 0 : kk)];
        const C2<T> zc = cconj<T>(Z[r * ld + (kk == 0 ? 0 : M - kk)]);
        const C2<T> E = cmk<T>(T(0.5) * (zk.x + zc.x), T(0.5) * (zk.y + zc.y));
        // O = (zk - zc) / (2i) = (-i/2)(zk - zc)
        const C2<T> d = csub<T>(zk, zc);
        const C2<T> O = cmk<T>(T(0.5) * d.y, T(-0.5) * d.x);
        A.S[(int64_t)row * A.Ms + kk] = cadd<T>(E, cmul<T>(A.post[kk], O));
    }
}

// ---------------------------------------------------------------------------------------------
// X-backward: C2R along x, writes out[i, j, k] = x / n_norm (+ optional mean subtraction)
// ---------------------------------------------------------------------------------------------
template <class T> struct XBwdArgs {
    DevGrid<T> g;
    const C2<T> *S;
    const C2<T> *tw;
    const FftStage *stages;
    const C2<T> *post;
    T *out;            // field interior view (strided) or dense array
    int dense;
    T scale;           // 1 / (Nx · Ny · Nz-normalisations)
    StepScalar<T> divisor;   // the written value is (x · scale) / divisor
    // even Nx: take X_0 and X_{Nx/2} as real, which they are but for rounding.  Their imaginary parts
    // hold the forward passes' rounding, amplified at the longest y and z waves by the inverse
    // Laplacian, and would enter the output as a ±1 wave along x (a u error of 4e-6 of max |u| at
    // 16 × 16 × 300 in FP32, 5e-7 without).  On with XFwdArgs::compensated.
    int real_ends;
    LineGeom L;
    FastDiv fNy;
    int Ms;
};

template <class T, bool MIXED> struct KXBwd {
    using Family = KXBwd<T, false>;   // one kernel of the step: a batch may hold both variants
    static constexpr int kThreads = kFftThreads, kMinBlocks = 1;
    static __device__ __forceinline__ void run(const XBwdArgs<T> &A, const Blk &B);
};
template <class T, bool MIXED> __device__ __forceinline__ void KXBwd<T, MIXED>::run(const XBwdArgs<T> &A, const Blk &B) {
    extern __shared__ unsigned char smem_raw[];
    const T divisor = A.divisor.get();
    const int Nx = A.g.Nx, Ny = A.g.Ny;
    const bool half = (Nx & 1) == 0;
    const int M = half ? Nx / 2 : Nx;
    const int Mx = Nx / 2 + 1;
    const int R = A.L.R, ld = A.L.ld;
    C2<T> *twl = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *a = twl + M;
    C2<T> *b = a + R * ld;
    const int row0 = B.x * R;
    const int nrows = Ny * A.g.Nz;
    load_table<T>(twl, A.tw, M);
    // blockDim.x / R threads per row, as in k_xfwd: a thread's row and its addresses are fixed
    const int lgt = __builtin_ctz((unsigned)blockDim.x) - A.L.lgR;   // log2 of threads per row
    const int tpr = 1 << lgt;
    const int r = threadIdx.x >> lgt, l = threadIdx.x & (tpr - 1);
    const int row = row0 + r;
    const bool live = row < nrows;
    {
        const C2<T> *Srow = A.S + (int64_t)(live ? row : 0) * A.Ms;
        constexpr int B = 4;
        for (int k0 = l; k0 < M; k0 += B * tpr) {
            C2<T> v[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int kk = k0 + u * tpr;
                C2<T> Zk = cmk<T>(T(0), T(0));
                if (live && kk < M) {
                    if (!half) {
                        Zk = kk < Mx ? Srow[kk] : cconj<T>(Srow[Nx - kk]);
                    } else {
                        C2<T> Xk = Srow[kk];
                        C2<T> Xc = cconj<T>(Srow[M - kk]);
                        if (kk == 0 && A.real_ends) Xk.y = Xc.y = T(0);
                        const C2<T> E = cmk<T>(T(0.5) * (Xk.x + Xc.x), T(0.5) * (Xk.y + Xc.y));
                        const C2<T> d = csub<T>(Xk, Xc);
                        // O = (Xk - conj(X_{M-k})) · e^{+2πik/N} / 2 ;  Z = E + i O
                        const C2<T> O = cmul<T>(cmk<T>(T(0.5) * d.x, T(0.5) * d.y), cconj<T>(A.post[kk]));
                        Zk = cmk<T>(E.x - O.y, E.y + O.x);
                    }
                }
                v[u] = Zk;
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int kk = k0 + u * tpr;
                if (kk < M) a[r * ld + kk] = v[u];
            }
        }
    }
    __syncthreads();
    const C2<T> *z = lds_fft<T, MIXED>(a, b, R, M, ld, twl, true, A.stages);
    if (live) {
        const int k = (int)fdiv((uint32_t)row, A.fNy), j = row - k * Ny;
        T *dst = A.dense ? A.out + (int64_t)Nx * ((int64_t)j + (int64_t)Ny * k) : A.out + idx3(0, j, k, A.g.sy, A.g.sz);
        for (int i = l; i < Nx; i += tpr) {
            T x;
            if (half) { const C2<T> zz = z[r * ld + (i >> 1)]; x = (i & 1) ? zz.y : zz.x; }
            else x = z[r * ld + i].x;
            dst[i] = ft_div<T>(x * A.scale, divisor);   // IEEE in FP64; FP32 by the reciprocal of the divisor
        }
    }
}

// −v / den, and 0 for the zero mode
template <class T> __device__ __forceinline__ C2<T> eig_divide(C2<T> v, T den, bool zero_mode) {
    return zero_mode ? cmk<T>(T(0), T(0)) : cmk<T>(ft_div<T>(-v.x, den), ft_div<T>(-v.y, den));
}

// ---------------------------------------------------------------------------------------------
// Y pass: complex FFT along y.  Lines ℓ = k·Ms + kx (ℓ < Ms·Nz, Ms the padded row stride), R
// consecutive lines per block; element j of line ℓ sits at S[(k·Ny + j)·Ms + kx].  Lines with
// kx ≥ Mx are row padding and are skipped.
// fused_divide: forward → divide by eigenvalues → backward (y is the last non-Flat axis).
// ---------------------------------------------------------------------------------------------
template <class T> struct YArgs {
    DevGrid<T> g;
    C2<T> *S;
    const C2<T> *tw;
    const FftStage *stages;
    int Mx, Ms;
    int inverse;
    int fused_divide;
    const T *lx, *ly;   // eigenvalues (fused)
    LineGeom L;
    FastDiv fMs;        // division by the row stride Ms
};

template <class T, bool MIXED> struct KYPass {
    using Family = KYPass<T, false>;   // one kernel of the step: a batch may hold both variants
    static constexpr int kThreads = kFftThreads, kMinBlocks = 1;
    static __device__ __forceinline__ void run(const YArgs<T> &A, const Blk &B);
};
template <class T, bool MIXED> __device__ __forceinline__ void KYPass<T, MIXED>::run(const YArgs<T> &A, const Blk &B) {
    extern __shared__ unsigned char smem_raw[];
    const int Ny = A.g.Ny, Mx = A.Mx, R = A.L.R, lgR = A.L.lgR, ld = A.L.ld;
    C2<T> *twl = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *a = twl + Ny;
    C2<T> *b = a + R * ld;
    const int Ms = A.Ms;
    const int nlines = Ms * A.g.Nz;
    // blockDim.x is a multiple of R, so every element a thread stages belongs to the same line
    const int r = threadIdx.x & (R - 1);
    const int line = B.x * R + r;
    const int k = (int)fdiv((uint32_t)line, A.fMs), kx = line - k * Ms;
    const bool valid = line < nlines && kx < Mx;                         // padding lines: nothing
    C2<T> *col = A.S + (int64_t)k * Ny * Ms + kx;
    load_table<T>(twl, A.tw, Ny);
    staged_copy<8>(R * Ny,
        [&](int t) { return valid ? col[(int64_t)(t >> lgR) * Ms] : cmk<T>(T(0), T(0)); },
        [&](int t, C2<T> v) { a[r * ld + (t >> lgR)] = v; });
    __syncthreads();
    C2<T> *res = lds_fft<T, MIXED>(a, b, R, Ny, ld, twl, A.inverse != 0, A.stages);
    if (A.fused_divide) {
        C2<T> *other = (res == a) ? b : a;
        for (int t = threadIdx.x; t < R * Ny; t += blockDim.x) {
            const int j = t >> lgR;
            if (valid) res[r * ld + j] = eig_divide<T>(res[r * ld + j], A.lx[kx] + A.ly[j], kx == 0 && j == 0);
        }
        __syncthreads();
        res = lds_fft<T, MIXED>(res, other, R, Ny, ld, twl, true, A.stages);
    }
    if (!valid) return;
    for (int t = threadIdx.x; t < R * Ny; t += blockDim.x) {
        const int j = t >> lgR;
        col[(int64_t)j * Ms] = res[r * ld + j];
    }
}

// ---------------------------------------------------------------------------------------------
// Z pass (last axis): forward transform, eigenvalue division, backward transform.  Lines
// ℓ = j·Ms + kx (ℓ < Ms·Ny), R consecutive lines per block; element k of line ℓ sits at
// S[k·Ny·Ms + ℓ], so a block reads R contiguous values per level; lines with kx ≥ Mx are row
// padding and are skipped.
//   zmode 0 (Periodic z): FFT of length Nz.
//   zmode 1 (Bounded z): the DCT-II of length N = Nz through one complex FFT of length N
//     (Makhoul 1980): v = (x0, x2, x4, …, x5, x3, x1), V = FFT(v),
//     X_k = c_k V_k + c̄_k V_{N−k} with c_k = e^{−iπk/2N}; after the division the inverse is
//     V'_k = c̄_k (Φ_k − i Φ_{N−k}) (Φ_N = 0), v' = IFFT(V'), x read back through the same
//     permutation.  Each thread handles the pair (k, N−k).  The result equals the inverse
//     transform of the 2N-point even extension, so it shares that normalisation (1 / 2N).  For odd
//     N every k > 0 has a partner other than itself.
// ---------------------------------------------------------------------------------------------
template <class T> struct ZArgs {
    DevGrid<T> g;
    C2<T> *S;
    const C2<T> *tw;         // table for the FFT length Nz
    const FftStage *stages;
    const C2<T> *dct;        // c_k, k < Nz (zmode 1)
    int Mx, Ms, zmode;       // Ms: row stride of S
    const T *lx, *ly, *lz;   // lz: Nz entries (Periodic), 2Nz (Bounded, symmetric)
    LineGeom G;
};

template <class T, bool MIXED> struct KZPass {
    using Family = KZPass<T, false>;   // one kernel of the step: a batch may hold both variants
    static constexpr int kThreads = kFftThreads, kMinBlocks = 1;
    static __device__ __forceinline__ void run(const ZArgs<T> &A, const Blk &B);
};
template <class T, bool MIXED> __device__ __forceinline__ void KZPass<T, MIXED>::run(const ZArgs<T> &A, const Blk &B) {
    extern __shared__ unsigned char smem_raw[];
    const int Ny = A.g.Ny, Nz = A.g.Nz, L = Nz, Mx = A.Mx, zmode = A.zmode;
    const int R = A.G.R, lgR = A.G.lgR, ld = A.G.ld;
    C2<T> *twl = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *dctl = twl + L;
    C2<T> *a = dctl + (zmode == 1 ? Nz : 0);
    C2<T> *b = a + R * ld;
    const int Ms = A.Ms;
    const int nlines = Ms * Ny;
    const int r = threadIdx.x & (R - 1);   // blockDim.x is a multiple of R
    const int line = B.x * R + r;
    const int j = line < nlines ? line / Ms : 0, kx = line - j * Ms;
    const bool valid = line < nlines && kx < Mx;   // padding lines: nothing
    const int64_t plane = (int64_t)Ny * Ms;
    C2<T> *col = A.S + line;
    load_table<T>(twl, A.tw, L);
    if (zmode == 1) load_table<T>(dctl, A.dct, Nz);
    staged_copy<8>(R * Nz,
        [&](int t) { return valid ? col[(int64_t)(t >> lgR) * plane] : cmk<T>(T(0), T(0)); },
        [&](int t, C2<T> v) {
            const int k = t >> lgR;
            a[r * ld + (zmode == 1 ? ((k & 1) ? Nz - ((k + 1) >> 1) : (k >> 1)) : k)] = v;
        });
    __syncthreads();
    C2<T> *res = lds_fft<T, MIXED>(a, b, R, L, ld, twl, false, A.stages);
    C2<T> *other = (res == a) ? b : a;
    const T lxy = valid ? A.lx[kx] + A.ly[j] : T(1);
    const bool zero_col = kx == 0 && j == 0;
    if (zmode == 1) {
        const int hN = Nz >> 1;
        for (int t = threadIdx.x; t < R * (hN + 1); t += blockDim.x) {
            const int kk = t >> lgR, p = kk == 0 ? 0 : Nz - kk;
            C2<T> *row = res + r * ld;
            const C2<T> Vk = row[kk], Vp = row[p];
            const C2<T> ck = dctl[kk], cp = dctl[p];
            const C2<T> Xk = cadd<T>(cmul<T>(ck, Vk), cmul<T>(cconj<T>(ck), Vp));
            const C2<T> Xp = cadd<T>(cmul<T>(cp, Vp), cmul<T>(cconj<T>(cp), Vk));
            const C2<T> Fk = eig_divide<T>(Xk, lxy + A.lz[kk], zero_col && kk == 0);
            const C2<T> Fp = kk == 0 ? cmk<T>(T(0), T(0)) : eig_divide<T>(Xp, lxy + A.lz[p], false);
            // V'_k = c̄_k (Φ_k − i Φ_{N−k}),  −i·z = (z.y, −z.x)
            row[kk] = cmul<T>(cconj<T>(ck), cmk<T>(Fk.x + Fp.y, Fk.y - Fp.x));
            if (p != kk) row[p] = cmul<T>(cconj<T>(cp), cmk<T>(Fp.x + Fk.y, Fp.y - Fk.x));
        }
    } else {
        for (int t = threadIdx.x; t < R * L; t += blockDim.x) {
            const int k = t >> lgR;
            res[r * ld + k] = eig_divide<T>(res[r * ld + k], lxy + A.lz[k], zero_col && k == 0);
        }
    }
    __syncthreads();
    res = lds_fft<T, MIXED>(res, other, R, L, ld, twl, true, A.stages);
    if (!valid) return;
    for (int t = threadIdx.x; t < R * Nz; t += blockDim.x) {
        const int k = t >> lgR;
        const int pos = zmode == 1 ? ((k & 1) ? Nz - ((k + 1) >> 1) : (k >> 1)) : k;
        col[(int64_t)k * plane] = res[r * ld + pos];
    }
}

// ---------------------------------------------------------------------------------------------
// Fourier–tridiagonal z solve per (kx, ky) column (diagonals from
// fourier_tridiagonal_poisson_solver.jl:199-229).  Two lanes of one wave share a column and eliminate
// towards its middle level, one from the bottom and one from the top; the middle level's equation
// closes the two chains and both substitute back outwards.  Columns ℓ = ky·Ms + kx are flattened, so that a level of a block's columns is one
// contiguous run (level k of column ℓ at k·(Ms·Ny) + ℓ; columns with kx ≥ Mx are row padding, never
// stored).  The chain's memory round trips bound it: a batch of tri_batch levels (16 FP32, 8 FP64) is
// loaded while the one before it is eliminated, and with KEEP the eliminated column stays in LDS (else,
// for columns too long for that, only its ratios do, and its values go through the spectrum's memory).
// The (0,0) column is singular, and the reference elides its last pivot: the top level's equation is
// the one that a source with a volume integral leaves unmet.  Here that level's source is replaced by
// what makes the column solvable, which has the same solution, and the closing pivot is elided;
// the constant this leaves is removed with the column mean (ϕ -= mean(ϕ), :253).  No other column
// loses a level: the reference's pivot guard (10·ε) is there for the rounding of a pivot that is a difference, and in
// FP32 it also takes the closing level of every column with λ · depth below 1e-6 (a 100 m layer over
// 2000 km) and with it the column's solution; here pivots are sums of positive numbers.
// ---------------------------------------------------------------------------------------------
template <class T> struct TriArgs {
    DevGrid<T> g;
    C2<T> *S;
    int Mx, Ms;
    const T *lx, *ly;
};
// whether a closing pivot can be divided by (0 in the singular column)
template <class T> __device__ __forceinline__ bool closes(T pivot) { return pivot >= std::numeric_limits<T>::min(); }

template <class T> constexpr int tri_batch() { return sizeof(T) == 4 ? 16 : 8; }
// LDS bytes of a block of bw columns
template <class T> constexpr size_t tri_lds(int Nz, int bw, bool keep) {
    return ((size_t)Nz * bw * (keep ? 3 : 1) + (keep ? 2 * (size_t)Nz + 1 : 0)) * sizeof(T);
}

template <class T, bool KEEP>
__global__ void __launch_bounds__(64) k_tridiag(TriArgs<T> A, C2<T> *__restrict__ Sg, const T *__restrict__ dzc,
                                                const T *__restrict__ idzf) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    constexpr int KB = tri_batch<T>();
    const int Ny = A.g.Ny, Nz = A.g.Nz, Mx = A.Mx;
    const int bw = blockDim.x >> 1;            // columns of the block
    C2<T> *ph = reinterpret_cast<C2<T> *>(smem_raw);                  // KEEP: [Nz][bw]
    T *tt = reinterpret_cast<T *>(ph + (KEEP ? (size_t)Nz * bw : 0));   // [Nz][bw]
    T *dz = tt + (size_t)Nz * bw;              // KEEP: [Nz] Δzᶜ
    T *iz = dz + Nz;                           // and [Nz + 1] 1/Δzᶠ, the end faces 0
    auto spacing = [&](int k) -> T { return KEEP ? dz[k] : dzc[k]; };
    auto coupling = [&](int k) -> T { return KEEP ? iz[k] : (k == 0 || k == Nz ? T(0) : idzf[k]); };
    const bool down = (int)threadIdx.x >= bw;   // this lane's chain: from the top
    const int c = threadIdx.x - (down ? bw : 0);
    const int64_t ncol = (int64_t)A.Ms * Ny;
    const int64_t col = min((int64_t)blockIdx.x * bw + c, ncol - 1);   // (lanes past the end repeat the last)
    const int j = (int)(col / A.Ms), kx = min((int)(col - (int64_t)j * A.Ms), Mx - 1);
    const bool store = (int64_t)blockIdx.x * bw + c == col && col - (int64_t)j * A.Ms < Mx;
    const T lam = A.lx[kx] + A.ly[j];

    C2<T> *S = Sg + col;
    const int mid = Nz >> 1;                        // the closing level
    const int steps = down ? Nz - 1 - mid : mid;    // levels of this chain
    const int longest = mid, common = Nz - 1 - mid;
    auto level = [&](int q) -> int { return down ? Nz - 1 - q : q; };
    auto at = [&](int k) -> int64_t { return (int64_t)k * ncol; };
    // a chain longer than its column's half reads a level of the other half, and drops it
    auto load = [&](C2<T> (&f)[KB], int q0) {
#pragma unroll
        for (int u = 0; u < KB; ++u) f[u] = S[at(level(min(q0 + u, longest)))];
    };
    // The chain carries each pivot as −(next + excess), where excess = Δz·λ + before·excess_prev / (before +
    // excess_prev) collects what exceeds the couplings: sums and products of positive numbers, so the
    // nearly singular columns of the longest waves keep the whole precision that the differences of a
    // pivot's recurrence lose.
    // (ft_div: IEEE division in FP64; the hardware reciprocal in FP32, which shortens the serial chain)
    T excess = T(0);
    T ratio = T(0);                    // coupling / −pivot of the chain's last level
    C2<T> phi = cmk<T>(T(0), T(0));    // its right-hand side / pivot
    // level q with couplings `before` (towards the chain's start) and `next`, and spacing d
    auto eliminate = [&](int q, const C2<T> &f, T before, T next, T d) {
        const int k = level(q);
        excess = d * lam + excess * ratio;
        const T pivot = next + excess;
        ratio = ft_div<T>(next, pivot);
        phi = cmk<T>(ft_div<T>(before * phi.x - f.x, pivot), ft_div<T>(before * phi.y - f.y, pivot));
        tt[k * bw + c] = ratio;
        if (KEEP) ph[k * bw + c] = phi;
        else if (store) S[at(k)] = phi;
    };
    const C2<T> fmid = S[at(mid)];
    C2<T> f[KB];
    load(f, 0);
    if (KEEP) {
        for (int k = threadIdx.x; k < Nz; k += blockDim.x) {
            dz[k] = dzc[k];
            iz[k] = k == 0 ? T(0) : idzf[k];
        }
        if (threadIdx.x == 0) iz[Nz] = T(0);
    }
    __syncthreads();
    const bool singular = lam == T(0);   // the (0,0) column
    if (blockIdx.x == 0) {
        C2<T> below = cmk<T>(T(0), T(0));   // (its source without the top level, summed by the whole wave)
        for (int k = threadIdx.x; k < Nz - 1; k += blockDim.x) below = cadd<T>(below, Sg[at(k)]);
        for (int o = bw; o > 0; o >>= 1) below = cadd<T>(below, cmk<T>(__shfl_xor(below.x, o), __shfl_xor(below.y, o)));
        if (singular && down) f[0] = cmk<T>(-below.x, -below.y);
    }
    for (int q0 = 0; q0 < longest; q0 += KB) {
        C2<T> nxt[KB];
        load(nxt, q0 + KB);   // (also beyond the end, repeating a level: where a branch could have left these loads out, the
                              // waits for the batch at hand would wait for them)
        // (the batch's coefficients before its arithmetic, whose stores to LDS they could not pass)
        T w[KB + 1], d[KB];
#pragma unroll
        for (int u = 0; u <= KB; ++u) w[u] = coupling(down ? Nz - min(q0 + u, Nz) : min(q0 + u, Nz));
#pragma unroll
        for (int u = 0; u < KB; ++u) d[u] = spacing(level(min(q0 + u, longest)));
        if (q0 + KB <= common) {
#pragma unroll
            for (int u = 0; u < KB; ++u) eliminate(q0 + u, f[u], w[u], w[u + 1], d[u]);
        } else {
#pragma unroll
            for (int u = 0; u < KB; ++u)
                if (q0 + u < steps) eliminate(q0 + u, f[u], w[u], w[u + 1], d[u]);
        }
#pragma unroll
        for (int u = 0; u < KB; ++u) f[u] = nxt[u];
    }
    // the closing level: its neighbours' chains end in (excess, ratio, phi) of the two lanes
    C2<T> x;
    {
        const T eb = __shfl(excess, c) * __shfl(ratio, c), et = __shfl(excess, c + bw) * __shfl(ratio, c + bw);
        const C2<T> pb = cmk<T>(__shfl(phi.x, c), __shfl(phi.y, c)), pt = cmk<T>(__shfl(phi.x, c + bw), __shfl(phi.y, c + bw));
        const T below = coupling(mid), above = coupling(mid + 1);
        const T pivot = spacing(mid) * lam + (eb + et);
        if (!singular && closes<T>(pivot))
            x = cmk<T>(ft_div<T>((below * pb.x - fmid.x) + above * pt.x, pivot), ft_div<T>((below * pb.y - fmid.y) + above * pt.y, pivot));
        else x = cmk<T>(T(0), T(0));
    }
    C2<T> sum = down ? cmk<T>(T(0), T(0)) : x;
    if (store && !down) S[at(mid)] = x;
    auto fetch = [&](C2<T> (&p)[KB], int q0) {   // levels q0, q0 − 1, …
#pragma unroll
        for (int u = 0; u < KB; ++u) {
            const int k = level(max(q0 - u, 0));
            p[u] = KEEP ? ph[k * bw + c] : S[at(k)];
        }
    };
    // q runs down from longest − 1; a chain one level shorter skips the first
    for (int q0 = longest - 1; q0 >= 0; q0 -= KB) {
        C2<T> p[KB];
        T t[KB];
        fetch(p, q0);
#pragma unroll
        for (int u = 0; u < KB; ++u) t[u] = tt[level(max(q0 - u, 0)) * bw + c];
        // (stored together: a test a level would part the chain)
        if (q0 - KB + 1 >= 0 && q0 < common) {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                x = cmk<T>(p[u].x + t[u] * x.x, p[u].y + t[u] * x.y);
                sum = cadd<T>(sum, x);
                p[u] = x;
            }
            if (store) {
#pragma unroll
                for (int u = 0; u < KB; ++u) S[at(level(q0 - u))] = p[u];
            }
        } else {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                const int q = q0 - u;
                if (q >= 0 && q < steps) {
                    x = cmk<T>(p[u].x + t[u] * x.x, p[u].y + t[u] * x.y);
                    sum = cadd<T>(sum, x);
                    if (store) S[at(level(q))] = x;
                }
            }
        }
    }
    sum = cadd<T>(sum, cmk<T>(__shfl_xor(sum.x, bw), __shfl_xor(sum.y, bw)));
    if (singular && store) {
        // remove the mean of the (0,0) column: equals removing the volume mean of ϕ (the reference
        // subtracts the mean of the real field).  Each lane revisits the levels it stored, in batches
        // (one round trip per level would set the kernel's duration).
        const C2<T> m = cmk<T>(sum.x / T(Nz), sum.y / T(Nz));
        if (!down) S[at(mid)] = csub<T>(S[at(mid)], m);
        int q = 0;
        for (; q + KB <= steps; q += KB) {
            C2<T> v[KB];
#pragma unroll
            for (int u = 0; u < KB; ++u) v[u] = S[at(level(q + u))];
#pragma unroll
            for (int u = 0; u < KB; ++u) S[at(level(q + u))] = csub<T>(v[u], m);
        }
        for (; q < steps; ++q) S[at(level(q))] = csub<T>(S[at(level(q))], m);
    }
}

// The same solve for columns of up to 2·NR + 1 levels, held in registers from the loads, all issued at once,
// to the stores: no LDS but the levels' coefficients, so that every column of the grid is under way together.
// Both chains end at position NR − 1, next to the closing level, and start where their length says; the
// positions before hold nothing (no source, no coupling to the first level), so that the chains run without a
// branch.  256 × 256 × 128 FP32: 54 µs by one lane a column through memory, 40 µs by k_tridiag (its columns in
// LDS leave a second, half-empty round of blocks, and a batch's loads only the arithmetic of one batch to
// arrive in), 19 µs here, 3.9 TB/s of the spectrum in and out.  The recurrence of the excess takes the
// FP32 solution's error against FP64 from 1.3e-5 to 1.3e-6 (geometric mean over eight grids).
template <class T, int NR>
__global__ void __launch_bounds__(64, 2) k_tridiag_short(TriArgs<T> A, C2<T> *__restrict__ Sg, const T *__restrict__ dzc,
                                                      const T *__restrict__ idzf) {
    __shared__ __attribute__((aligned(16))) T before[2][NR], next[2][NR], dz[2][NR];   // by chain and position
    constexpr int bw = 32;                     // columns of the block
    const int Ny = A.g.Ny, Nz = A.g.Nz, Mx = A.Mx;
    const int down = threadIdx.x >= bw;
    const int c = threadIdx.x & (bw - 1);
    const int64_t ncol = (int64_t)A.Ms * Ny;
    const int64_t col = min((int64_t)blockIdx.x * bw + c, ncol - 1);
    const int j = (int)(col / A.Ms), kx = min((int)(col - (int64_t)j * A.Ms), Mx - 1);
    const bool store = (int64_t)blockIdx.x * bw + c == col && col - (int64_t)j * A.Ms < Mx;
    const T lam = A.lx[kx] + A.ly[j];
    C2<T> *S = Sg + col;
    const int mid = Nz >> 1;   // the closing level
    auto first_of = [&](int chain) -> int { return NR - (chain ? Nz - 1 - mid : mid); };
    auto level_of = [&](int chain, int q) -> int { return chain ? mid + NR - q : q - NR + mid; };
    const int first = first_of(down);
    auto at = [&](int k) -> int64_t { return (int64_t)k * ncol; };
    const C2<T> fmid = S[at(mid)];
    C2<T> f[NR];
    T t[NR];
    // the chain's first level (or the closing one) and the step to the next: one running address, formed anew
    // for the stores, instead of one a level kept from the loads
    C2<T> *line = S + at(level_of(down, first));
    const int64_t step = down ? -ncol : ncol;
    {
        const C2<T> *p = line;
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            f[q] = *p;
            p += q >= first ? step : 0;
        }
    }
    for (int e = threadIdx.x; e < 2 * NR; e += 64) {
        const int chain = e >= NR, q = e - (chain ? NR : 0), k = level_of(chain, q);
        const bool real = q >= first_of(chain);
        // (up: from the face below to the face above; down: the reverse)
        const T lo = real && k > 0 ? idzf[k] : T(0), hi = real && k < Nz - 1 ? idzf[k + 1] : T(0);
        before[chain][q] = chain ? hi : lo;
        next[chain][q] = real ? (chain ? lo : hi) : T(1);
        dz[chain][q] = real ? dzc[k] : T(0);
    }
    __syncthreads();
    const bool singular = lam == T(0);   // the (0,0) column
    C2<T> top = cmk<T>(T(0), T(0));
    if (blockIdx.x == 0) {   // (its source without the top level, summed by the whole wave)
        for (int k = threadIdx.x; k < Nz - 1; k += 64) top = csub<T>(top, Sg[at(k)]);
        for (int o = 32; o > 0; o >>= 1) top = cadd<T>(top, cmk<T>(__shfl_xor(top.x, o), __shfl_xor(top.y, o)));
    }
    const bool replace = singular && down;
    T excess = T(0), ratio = T(0);
    C2<T> phi = cmk<T>(T(0), T(0));
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        // (the pivots do not wait for the loads; but running far ahead they cost more registers
        // than the chain's values leave)
        if (q % (sizeof(T) == 4 ? 8 : 4) == 0) asm volatile("" : "+v"(excess), "+v"(ratio), "+v"(phi.x), "+v"(phi.y));
        C2<T> s = f[q];
        if (replace && q == first) s = top;
        if (q < first) s = cmk<T>(T(0), T(0));
        excess = dz[down][q] * lam + excess * ratio;
        const T pivot = next[down][q] + excess;
        ratio = ft_div<T>(next[down][q], pivot);
        phi = cmk<T>(ft_div<T>(before[down][q] * phi.x - s.x, pivot), ft_div<T>(before[down][q] * phi.y - s.y, pivot));
        f[q] = phi;
        t[q] = ratio;
    }
    C2<T> x;
    {
        // (a chain without levels couples to nothing)
        const T below = mid > 0 ? idzf[mid] : T(0), above = mid < Nz - 1 ? idzf[mid + 1] : T(0);
        const T eb = __shfl(excess, c) * __shfl(ratio, c), et = __shfl(excess, c + bw) * __shfl(ratio, c + bw);
        const C2<T> pb = cmk<T>(__shfl(phi.x, c), __shfl(phi.y, c)), pt = cmk<T>(__shfl(phi.x, c + bw), __shfl(phi.y, c + bw));
        const T pivot = dzc[mid] * lam + (eb + et);
        if (!singular && closes<T>(pivot))
            x = cmk<T>(ft_div<T>((below * pb.x - fmid.x) + above * pt.x, pivot), ft_div<T>((below * pb.y - fmid.y) + above * pt.y, pivot));
        else x = cmk<T>(T(0), T(0));
    }
    const C2<T> xmid = x;
    C2<T> sum = down ? cmk<T>(T(0), T(0)) : x;
#pragma unroll
    for (int q = NR - 1; q >= 0; --q) {
        x = cmk<T>(f[q].x + t[q] * x.x, f[q].y + t[q] * x.y);
        f[q] = x;
        if (q >= first) sum = cadd<T>(sum, x);
    }
    sum = cadd<T>(sum, cmk<T>(__shfl_xor(sum.x, bw), __shfl_xor(sum.y, bw)));
    // the (0,0) column without its mean: equals removing the volume mean of ϕ
    const C2<T> mean = singular ? cmk<T>(sum.x / T(Nz), sum.y / T(Nz)) : cmk<T>(T(0), T(0));
    if (!store) return;
    if (!down) S[at(mid)] = csub<T>(xmid, mean);
    asm volatile("" : "+v"(line));
#pragma unroll
    for (int q = 0; q < NR; ++q)
        if (q >= first) {
            *line = csub<T>(f[q], mean);
            line += step;
        }
}

// ---------------------------------------------------------------------------------------------
// FP64 iterative refinement: residual of a computed solution and the correction update
// ---------------------------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(256) k_poisson_residual(Ctx<T> C, RefineOp L, const T *p, int64_t psy, int64_t psz,
                                                          const double *b64, StepScalar<T> divisor, T *r) {
    const DevGrid<T> &g = C.g;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= g.Nx || j >= g.Ny) return;
    const int64_t dense = (int64_t)i + (int64_t)g.Nx * ((int64_t)j + (int64_t)g.Ny * k);
    const int ip = i + 1 == g.Nx ? 0 : i + 1, im = i == 0 ? g.Nx - 1 : i - 1;
    const int jp = j + 1 == g.Ny ? 0 : j + 1, jm = j == 0 ? g.Ny - 1 : j - 1;
    double b;
    if (b64) b = b64[dense];
    else {
        // ∇·U in FP64 from the stored velocities (divergence_operators.jl:16-19 on a rectilinear grid)
        b = 0;
        if (!C.flx()) b += ((double)C.ld(C.s.U[0], ip, j, k) - (double)C.ld(C.s.U[0], i, j, k)) * (double)g.idx;
        if (!C.fly()) b += ((double)C.ld(C.s.U[1], i, jp, k) - (double)C.ld(C.s.U[1], i, j, k)) * (double)g.idy;
        if (!C.flz())
            b += ((double)C.ld(C.s.U[2], i, j, k + 1) - (double)C.ld(C.s.U[2], i, j, k)) * (L.ihz2 < 0 ? L.idzc[k] : (double)g.idzc[k]);
        b *= 1.0 / (double)divisor.get();
    }
    auto P = [&](int ii, int jj, int kk) -> double { return (double)p[(int64_t)ii + psy * jj + psz * kk]; };
    const double pc = P(i, j, k);
    double lap = 0;
    if (!C.flx()) lap += ((P(ip, j, k) - pc) - (pc - P(im, j, k))) * L.ihx2;
    if (!C.fly()) lap += ((P(i, jp, k) - pc) - (pc - P(i, jm, k))) * L.ihy2;
    if (!C.flz()) {
        const bool per = g.tz == OM_PERIODIC;
        const int kp = k + 1 == g.Nz ? (per ? 0 : -1) : k + 1, km = k == 0 ? (per ? g.Nz - 1 : -1) : k - 1;
        if (L.ihz2 >= 0) {
            const double up = kp >= 0 ? P(i, j, kp) - pc : 0.0, dn = km >= 0 ? pc - P(i, j, km) : 0.0;
            lap += (up - dn) * L.ihz2;
        } else {   // stretched: (flux through face k+1 − flux through face k) / Δzᶜ
            const double up = kp >= 0 ? (P(i, j, kp) - pc) * L.idzf[k + 1] : 0.0;
            const double dn = km >= 0 ? (pc - P(i, j, km)) * L.idzf[k] : 0.0;
            lap += (up - dn) * L.idzc[k];
        }
    }
    r[dense] = (T)(b - lap);
}

template <class T>
__global__ void __launch_bounds__(256) k_add_correction(DevGrid<T> g, T *p, int64_t psy, int64_t psz, const T *d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= g.Nx || j >= g.Ny) return;
    p[(int64_t)i + psy * j + psz * k] += d[(int64_t)i + (int64_t)g.Nx * ((int64_t)j + (int64_t)g.Ny * k)];
}

template <class T> void launch_poisson_residual(const Ctx<T> &C, const RefineOp &L, const T *p, int64_t psy, int64_t psz,
                                                const double *b64, StepScalar<T> divisor, T *r, hipStream_t st) {
    const dim3 blk(64, 4, 1), grid((C.g.Nx + 63) / 64, (C.g.Ny + 3) / 4, C.g.Nz);
    hipLaunchKernelGGL(k_poisson_residual<T>, grid, blk, 0, st, C, L, p, psy, psz, b64, divisor, r);
}
template <class T> void launch_add_correction(const DevGrid<T> &g, T *p, int64_t psy, int64_t psz, const T *d, hipStream_t st) {
    const dim3 blk(64, 4, 1), grid((g.Nx + 63) / 64, (g.Ny + 3) / 4, g.Nz);
    hipLaunchKernelGGL(k_add_correction<T>, grid, blk, 0, st, g, p, psy, psz, d);
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
static int ilog2(int v) { int l = 0; while ((1 << l) < v) ++l; return l; }

// R lines of length n with `tables` complex table entries in front (om_kernels.h chooses R)
static LineGeom line_geom(int n, int tables, size_t e, size_t &lds) {
    const int R = fft_lines_per_block(n, tables, e);
    if (R < 1) throw std::runtime_error("FFT line does not fit in LDS");
    const int ld = R > 1 ? n + 1 : n;
    const bool p2 = (n & (n - 1)) == 0;
    lds = ((size_t)(p2 ? 1 : 2) * R * ld + tables) * e;
    return LineGeom{R, ilog2(R), ld};
}

template <class T> void launch_poisson(const PoissonPlan<T> &P, const Ctx<T> &C, const T *src, T *out, int dense_out,
                                       StepScalar<T> divisor, hipStream_t st) {
    const DevGrid<T> &g = C.g;
    const size_t e = sizeof(C2<T>);
    const size_t budget = 64 * 1024;
    const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
    const int M = (Nx & 1) == 0 ? Nx / 2 : Nx;
    const int Mx = Nx / 2 + 1;
    const int nrows = Ny * Nz;
    size_t lds = 0;
    auto p2 = [](int n) { return (n & (n - 1)) == 0; };
    const int compensated = !(p2(M) && p2(Ny) && (P.tridiagonal || p2(Nz)));
    // one of a kernel's two variants by its line length
    auto by_length = [&](auto plain, auto mixed, int n, int blocks, size_t shared, const auto &A) {
        if (p2(n)) launch_k<decltype(plain)>(dim3(blocks), dim3(kFftThreads), shared, st, A);
        else launch_k<decltype(mixed)>(dim3(blocks), dim3(kFftThreads), shared, st, A);
    };
    {
        const LineGeom L = line_geom(M, M, e, lds);
        XFwdArgs<T> A{C, src, P.S, P.tw_xh, P.st_x, P.post, P.tridiagonal, compensated, L, make_fastdiv((uint32_t)Ny), make_fastdiv((uint32_t)Mx), P.Ms};
        const int blocks = (nrows + L.R - 1) / L.R;
        if (src) by_length(KXFwd<T, false, kSrcDense>(), KXFwd<T, true, kSrcDense>(), M, blocks, lds, A);
        else if (poisson_source_reads_no_halo(C)) by_length(KXFwd<T, false, kSrcVelocity>(), KXFwd<T, true, kSrcVelocity>(), M, blocks, lds, A);
        else by_length(KXFwd<T, false, kSrcGeneral>(), KXFwd<T, true, kSrcGeneral>(), M, blocks, lds, A);
    }
    const bool z_active = g.tz != OM_FLAT;
    const LineGeom Ly = line_geom(Ny, Ny, e, lds);
    const size_t lds_y = lds;
    const int ygrid = (P.Ms * Nz + Ly.R - 1) / Ly.R;
    {
        YArgs<T> A{g, P.S, P.tw_y, P.st_y, Mx, P.Ms, 0, z_active ? 0 : 1, P.lx, P.ly, Ly, make_fastdiv((uint32_t)P.Ms)};
        by_length(KYPass<T, false>(), KYPass<T, true>(), Ny, ygrid, lds_y, A);
    }
    T scale = T(1) / (T(M) * T(Ny));
    if (z_active) {
        if (P.tridiagonal) {
            TriArgs<T> A{g, P.S, Mx, P.Ms, P.lx, P.ly};
            const int64_t ncol = (int64_t)P.Ms * Ny;
            const int half = Nz >> 1;
            // registers hold chains of up to 64 levels in FP32 (241 VGPRs, two waves a SIMD) and 32 in FP64 (247)
            constexpr int most = sizeof(T) == 4 ? 64 : 32;
            if (half <= most) {
                const auto kernel = half <= 16 ? &k_tridiag_short<T, 16> : (half <= 32 ? &k_tridiag_short<T, 32> : &k_tridiag_short<T, most>);
                hipLaunchKernelGGL(kernel, dim3((unsigned)((ncol + 31) / 32)), dim3(64), 0, st, A, P.S, g.dzc, g.idzf);
            } else {
                // columns per block (two lanes each, one wave, partly filled when narrow): each column is a
                // serial sweep, so the launch wants waves on every SIMD (≥ 2048 of them) more than full
                // waves; 16 columns still read whole 128-byte lines of the spectrum.
                int bw = 32;
                while (bw > 16 && ncol / bw < 2048) bw >>= 1;
                while (bw > 8 && tri_lds<T>(Nz, bw, true) > budget) bw >>= 1;
                const bool keep = tri_lds<T>(Nz, bw, true) <= budget;
                while (bw > 1 && tri_lds<T>(Nz, bw, keep) > budget) bw >>= 1;
                const auto kernel = keep ? &k_tridiag<T, true> : &k_tridiag<T, false>;
                hipLaunchKernelGGL(kernel, dim3((unsigned)((ncol + bw - 1) / bw)), dim3(2 * bw), tri_lds<T>(Nz, bw, keep), st, A, P.S, g.dzc,
                                   g.idzf);
            }
        } else {
            const LineGeom Lz = line_geom(Nz, z_line_tables(Nz, P.zmode == 1), e, lds);
            ZArgs<T> A{g, P.S, P.tw_z, P.st_z, P.tw_dct, Mx, P.Ms, P.zmode, P.lx, P.ly, P.lz, Lz};
            by_length(KZPass<T, false>(), KZPass<T, true>(), Nz, (P.Ms * Ny + Lz.R - 1) / Lz.R, lds, A);
            scale = T(1) / ((T(M) * T(Ny)) * T(P.Lz_norm));
        }
        YArgs<T> A{g, P.S, P.tw_y, P.st_y, Mx, P.Ms, 1, 0, P.lx, P.ly, Ly, make_fastdiv((uint32_t)P.Ms)};
        by_length(KYPass<T, false>(), KYPass<T, true>(), Ny, ygrid, lds_y, A);
    }
    {
        const LineGeom L = line_geom(M, M, e, lds);
        XBwdArgs<T> A{g, P.S, P.tw_xh, P.st_x, P.post, out, dense_out, scale, divisor, compensated, L, make_fastdiv((uint32_t)Ny), P.Ms};
        by_length(KXBwd<T, false>(), KXBwd<T, true>(), M, (nrows + L.R - 1) / L.R, lds, A);
    }
}

#ifndef OM_ONLY_DOUBLE
template void launch_poisson_residual<float>(const Ctx<float> &, const RefineOp &, const float *, int64_t, int64_t,
                                             const double *, StepScalar<float>, float *, hipStream_t);
template void launch_add_correction<float>(const DevGrid<float> &, float *, int64_t, int64_t, const float *, hipStream_t);
template void launch_poisson<float>(const PoissonPlan<float> &, const Ctx<float> &, const float *, float *, int, StepScalar<float>,
                                    hipStream_t);
#endif
#ifndef OM_ONLY_FLOAT
template void launch_poisson_residual<double>(const Ctx<double> &, const RefineOp &, const double *, int64_t, int64_t,
                                              const double *, StepScalar<double>, double *, hipStream_t);
template void launch_add_correction<double>(const DevGrid<double> &, double *, int64_t, int64_t, const double *, hipStream_t);
template void launch_poisson<double>(const PoissonPlan<double> &, const Ctx<double> &, const double *, double *, int, StepScalar<double>,
                                     hipStream_t);
#endif

}  // namespace om
