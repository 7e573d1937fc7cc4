// d2bi_integrate.cuh -- column integration: the stage-by-stage RK4 march and
// the shared step matrix for many precession points, in FP32 on the FAST field
// and in FP64.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ (c) integrate

// Points of one FAST integration launch, over all its fields, and the slots of
// their deviations (a wave of NP points may read NP - 1 past its field's last).
static constexpr int INT_POINTS = 32, INT_SLOTS = INT_POINTS + 31;

struct FastIntParams {
    int Mx, My, Mz, np;         // np: precession points per field
    int nsplit, split;          // waves per column, of them per field
    PointCount N;               // a field of no condition if over
    float b0, bg, dz;
    int64_t stride;             // records from one field to the next
    float aa[INT_SLOTS];        // 2 pi s_g per field and precession point
    float al[INT_SLOTS];        // 2 dz aa (the shared step matrix)
};

__device__ __forceinline__ float fm(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fm(double a, double b, double c) { return fma(a, b, c); }

// A pixel column of the FAST field: float4 {x, rho} with the density field,
// else float2 x (rho = 1); sample Mz is sample 0.  NT: non-temporal loads,
// where each sample is read once, keep the stream from displacing cached data.
template <bool DENS, bool NT>
struct FastColumn {
    typedef float4 Raw;
    const void* field;
    int64_t col, plane;
    int nz;
    float b0, bg;
    __device__ __forceinline__ Raw load(int k) const
    {
        const int64_t o = col + plane * (k == nz ? 0 : k);
        typedef float v2 __attribute__((ext_vector_type(2)));
        if (DENS) {
            // three words of the record: the fourth's register, free for other
            // use at once, would make that use wait for the load in flight (8
            // points: 73 us with three words, 85 with four)
            const float* f = static_cast<const float*>(field) + 4 * o;
            if (NT)
                return make_float4(__builtin_nontemporal_load(f), __builtin_nontemporal_load(f + 1),
                                   __builtin_nontemporal_load(f + 2), 0.0f);
            return make_float4(f[0], f[1], f[2], 0.0f);
        }
        const v2* f = static_cast<const v2*>(field) + o;
        const v2 v = NT ? __builtin_nontemporal_load(f) : *f;
        return make_float4(v.x, v.y, 1.0f, 0.0f);
    }
    __device__ __forceinline__ void coef(const Raw& f, float& c0, float& cgr, float& cgi) const
    {
        if (DENS) {
            c0 = b0 * f.z;
            const float bgr = bg * f.z;
            cgr = bgr * f.x;
            cgi = bgr * f.y;
        } else {
            c0 = b0;
            cgr = bg * f.x;
            cgi = bg * f.y;
        }
    }
};

// Points scaled by a power of two each, so that their largest component lies
// in [1/2, 1): no bit of what follows changes but the exponents.
template <int NP>
__device__ __forceinline__ void rescale(double* p0r, double* p0i, double* pgr, double* pgi)
{
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const double m = fmax(fmax(fabs(p0r[p]), fabs(p0i[p])), fmax(fabs(pgr[p]), fabs(pgi[p])));
        const int e = -__builtin_amdgcn_frexp_exp(m);
        p0r[p] = __builtin_amdgcn_ldexp(p0r[p], e);
        p0i[p] = __builtin_amdgcn_ldexp(p0i[p], e);
        pgr[p] = __builtin_amdgcn_ldexp(pgr[p], e);
        pgi[p] = __builtin_amdgcn_ldexp(pgi[p], e);
    }
}

// One lane per pixel column, NP precession points marched together from
// one read of the column (the field is shared by all precession points:
// precession changes s_g only).  Classic RK4 with h = 2 dz; the per-step
// renormalisation of the reference is a positive scalar on a linear map, so it
// is applied once at the end: I = |phi_g|^2/|phi|^2.  FP64 points are rescaled
// every `every` double steps (RS), so that a column of any depth and deviation
// stays in range; instances without are for those whose bound already does
// (rescale_every), and take no branch and no register for it.
// The mean-potential term c0 = b0 rho stays in, although in the exact ODE it
// is a global phase: RK4's truncation error depends on the whole matrix, and
// over 800 double steps leaving c0 out moves |phi_g|^2 by ~2e-4.
template <int NP, bool RS = false, class T, class S>
__device__ __forceinline__ void march_stage(const S& s, int nz, T dz, const T* aa, T* p0r, T* p0i, T* pgr, T* pgi,
                                            bool go, int every = 0)
{
    [[maybe_unused]] int left = every;
    const T dz3 = dz / 3, dz23 = 2 * dz / 3, dz2 = 2 * dz;
#pragma unroll
    for (int p = 0; p < NP; p++) { p0r[p] = 1; p0i[p] = 0; pgr[p] = 0; pgi[p] = 0; }
    // samples of the next PD double steps are in flight: ring[2u] and
    // ring[2u + 1] hold samples ii + 1, ii + 2 of the double step at ii in
    // slot u (ii = i0 + 2u), reloaded with those of ii + 2 PD once used.  A
    // column is a chain of dependent loads, so the depth, not the bandwidth,
    // bounds a wave's time when few points are marched per sample.
    constexpr int PD = NP <= 4 ? 4 : 1;
    T c0a = 0, cgra = 0, cgia = 0;
    typename S::Raw ring[2 * PD];
#pragma unroll
    for (int k = 0; k < 2 * PD; k++) ring[k] = typename S::Raw{};
    if (nz >= 2) {
        s.coef(s.load(0), c0a, cgra, cgia);
#pragma unroll
        for (int k = 0; k < 2 * PD; k++)
            if (k + 1 <= nz) ring[k] = s.load(k + 1);
    }
    for (int i0 = 0; go && i0 <= nz - 2; i0 += 2 * PD) {
#pragma unroll
    for (int u = 0; u < PD; u++) {
        const int ii = i0 + 2 * u;
        if (ii > nz - 2) break;
        T c0b, cgrb, cgib, c0c, cgrc, cgic;
        s.coef(ring[2 * u], c0b, cgrb, cgib);
        s.coef(ring[2 * u + 1], c0c, cgrc, cgic);
        if (ii + 2 * PD + 2 <= nz) {
            ring[2 * u] = s.load(ii + 2 * PD + 1);
            ring[2 * u + 1] = s.load(ii + 2 * PD + 2);
        }
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const T a = aa[p];
            T d0r, d0i, dgr, dgi;
#define FDERIV(c0, cgr, cgi)                                             \
    {                                                                    \
        const T ca_ = c0 + a;                                            \
        d0r = fm(-c0, p0i[p], fm(-cgi, pgr[p], -cgr * pgi[p]));          \
        d0i = fm(c0, p0r[p], fm(cgr, pgr[p], -cgi * pgi[p]));            \
        dgr = fm(cgi, p0r[p], fm(-cgr, p0i[p], -ca_ * pgi[p]));          \
        dgi = fm(cgr, p0r[p], fm(cgi, p0i[p], ca_ * pgr[p]));            \
    }
            const T s0r = p0r[p], s0i = p0i[p], sgr = pgr[p], sgi = pgi[p];
            FDERIV(c0a, cgra, cgia)
            T a0r = fm(d0r, dz3, s0r), a0i = fm(d0i, dz3, s0i);
            T agr = fm(dgr, dz3, sgr), agi = fm(dgi, dz3, sgi);
            p0r[p] = fm(d0r, dz, s0r); p0i[p] = fm(d0i, dz, s0i);
            pgr[p] = fm(dgr, dz, sgr); pgi[p] = fm(dgi, dz, sgi);
            FDERIV(c0b, cgrb, cgib)
            p0r[p] = fm(d0r, dz, s0r); p0i[p] = fm(d0i, dz, s0i);
            pgr[p] = fm(dgr, dz, sgr); pgi[p] = fm(dgi, dz, sgi);
            a0r = fm(d0r, dz23, a0r); a0i = fm(d0i, dz23, a0i);
            agr = fm(dgr, dz23, agr); agi = fm(dgi, dz23, agi);
            FDERIV(c0b, cgrb, cgib)
            p0r[p] = fm(d0r, dz2, s0r); p0i[p] = fm(d0i, dz2, s0i);
            pgr[p] = fm(dgr, dz2, sgr); pgi[p] = fm(dgi, dz2, sgi);
            a0r = fm(d0r, dz23, a0r); a0i = fm(d0i, dz23, a0i);
            agr = fm(dgr, dz23, agr); agi = fm(dgi, dz23, agi);
            FDERIV(c0c, cgrc, cgic)
#undef FDERIV
            p0r[p] = fm(d0r, dz3, a0r); p0i[p] = fm(d0i, dz3, a0i);
            pgr[p] = fm(dgr, dz3, agr); pgi[p] = fm(dgi, dz3, agi);
        }
        c0a = c0c; cgra = cgrc; cgia = cgic;
        if constexpr (RS) {
            if (--left == 0) {
                left = every;
                rescale<NP>(p0r, p0i, pgr, pgi);
            }
        }
    }
    }
}

// Sum of the first np points' |phi_g|^2 / |phi|^2.
template <int NP, class T>
__device__ __forceinline__ double intensity_sum(int np, const T* p0r, const T* p0i, const T* pgr, const T* pgi)
{
    double acc = 0.0;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        if (p >= np) break;
        const T ng = fm(pgr[p], pgr[p], pgi[p] * pgi[p]);
        const T n0 = fm(p0r[p], p0r[p], p0i[p] * p0i[p]);
        acc += (double)ng / (double)(n0 + ng);
    }
    return acc;
}

// Many precession points.  The system is phi' = i H(a) phi with
// H(a) = [[c0, cg], [conj(cg), c0 + a]] (the derivative above), so one RK4
// double step is phi <- M phi with
//     M = I + Q1/3 + (2/3) K2 + K3/3 + K4/6,
//     Q1 = dz A_a,  T1 = I + Q1,  K2 = dz A_b T1,  T2 = I + K2,
//     K3 = 2 dz A_b T2,  T3 = I + K3,  K4 = 2 dz A_c T3,   A_x = i H_x(a),
// the same map as the stage-by-stage march (A_a, A_b, A_c at the double
// step's three samples).  a enters only through the (2,2) element, once per
// stage, so the entries of M are polynomials in alpha = 2 dz a of degrees 2,
// 3, 3 and 4 whose coefficients depend on the column's field samples only.
// They are formed once per double step and shared: a precession point then
// costs a Horner evaluation at its alpha and one matrix-vector product
// (~40 FMAs) instead of four derivative evaluations and the stage updates
// (~80).  Results differ from the stage-by-stage march by rounding only.
template <class T>
struct cplx {
    T r, i;
};
template <int D, class T>
struct CPoly {
    cplx<T> c[D + 1];    // coefficients of alpha^0 .. alpha^D
};

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (B <= E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// Coefficients of one polynomial known to have no real (RE) or no imaginary
// part (IM): bit k for alpha^k.  alpha multiplies the (2,2) element by i alone,
// so the leading coefficients of the (2,2) entries are real or imaginary; an
// operation with the zero part would still be made (0 x is not 0 for every x).
template <unsigned RE, unsigned IM>
struct NoPart {
    static constexpr bool re(int k) { return (RE >> k) & 1u; }
    static constexpr bool im(int k) { return (IM >> k) & 1u; }
};

// One column (P1, P2) of Q = s A_x P for a polynomial matrix P, with the
// stage's scaled coefficients c = s c0, g = s cg and ax = s / (2 dz):
//     Q1 = i (c P1 + g P2),   Q2 = i (conj(g) P1 + c P2 + ax alpha P2).
// Terms are chained from the first present one, so structural zeros cost
// nothing; Z are the parts P2 lacks.
template <class Z, int D1, int D2, class T, int E1 = (D1 > D2 ? D1 : D2), int E2 = (D1 > D2 + 1 ? D1 : D2 + 1)>
__device__ __forceinline__ void rk_col(T c, T gr, T gi, T ax, const CPoly<D1, T>& P1, const CPoly<D2, T>& P2,
                                       CPoly<E1, T>& Q1, CPoly<E2, T>& Q2)
{
    static_for<0, E1>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        T ur, ui;
        if constexpr (k <= D2) {
            if constexpr (Z::re(k)) {
                ur = -gi * P2.c[k].i;
                ui = gr * P2.c[k].i;
            } else if constexpr (Z::im(k)) {
                ur = gr * P2.c[k].r;
                ui = gi * P2.c[k].r;
            } else {
                ur = fm(gr, P2.c[k].r, -gi * P2.c[k].i);
                ui = fm(gr, P2.c[k].i, gi * P2.c[k].r);
            }
            if constexpr (k <= D1) {
                ur = fm(c, P1.c[k].r, ur);
                ui = fm(c, P1.c[k].i, ui);
            }
        } else {
            ur = c * P1.c[k].r;
            ui = c * P1.c[k].i;
        }
        Q1.c[k] = cplx<T>{-ui, ur};
    });
    static_for<0, E2>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        constexpr bool ta = k <= D1, tb = k <= D2, tc = k >= 1 && k - 1 <= D2;
        constexpr bool br = tb && !Z::re(k), bi = tb && !Z::im(k);
        constexpr bool cr = tc && !Z::re(k - 1), ci = tc && !Z::im(k - 1);
        T ur = 0, ui = 0;
        if constexpr (ta) {
            ur = fm(gr, P1.c[k].r, gi * P1.c[k].i);
            ui = fm(gr, P1.c[k].i, -gi * P1.c[k].r);
        }
        if constexpr (br) ur = ta ? fm(c, P2.c[tb ? k : 0].r, ur) : c * P2.c[tb ? k : 0].r;
        if constexpr (bi) ui = ta ? fm(c, P2.c[tb ? k : 0].i, ui) : c * P2.c[tb ? k : 0].i;
        if constexpr (cr) ur = ta || br ? fm(ax, P2.c[tc ? k - 1 : 0].r, ur) : ax * P2.c[tc ? k - 1 : 0].r;
        if constexpr (ci) ui = ta || bi ? fm(ax, P2.c[tc ? k - 1 : 0].i, ui) : ax * P2.c[tc ? k - 1 : 0].i;
        Q2.c[k] = cplx<T>{-ui, ur};
    });
}

// M += s P (degree of P <= degree of M; Z: the parts P lacks)
template <class Z = NoPart<0, 0>, int DM, int DP, class T>
__device__ __forceinline__ void poly_axpy(CPoly<DM, T>& M, T s, const CPoly<DP, T>& P)
{
    static_assert(DP <= DM, "degree");
    static_for<0, DP>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr (!Z::re(k)) M.c[k].r = fm(s, P.c[k].r, M.c[k].r);
        if constexpr (!Z::im(k)) M.c[k].i = fm(s, P.c[k].i, M.c[k].i);
    });
}

// M at alpha (Z: parts its leading coefficient lacks)
template <class Z = NoPart<0, 0>, int D, class T>
__device__ __forceinline__ cplx<T> horner(const CPoly<D, T>& M, T al)
{
    cplx<T> v = M.c[D];
#pragma unroll
    for (int k = D - 1; k >= 0; k--) {
        v.r = fm(v.r, al, M.c[k].r);
        v.i = Z::im(D) && k == D - 1 ? M.c[k].i : fm(v.i, al, M.c[k].i);
    }
    return v;
}

// The column's march: NP points from (1, 0) through nz samples (sample nz is
// sample 0), or none if not go; S gives a sample's coefficients (load(k) what is read, coef(raw)
// c0 and cg).
template <int NP, bool RS = false, class T, class S>
__device__ __forceinline__ void march_poly(const S& s, int nz, T dz, const T* al_, T* p0r, T* p0i, T* pgr, T* pgi,
                                           bool go, int every = 0)
{
    [[maybe_unused]] int left = every;
    const T dz2 = 2 * dz, dz6 = dz / 3, third = T(1) / 3, two3 = T(2) / 3, sixth = T(1) / 6, half = T(0.5), one = T(1);
#pragma unroll
    for (int p = 0; p < NP; p++) { p0r[p] = 1; p0i[p] = 0; pgr[p] = 0; pgi[p] = 0; }
    // parts the leading coefficients of T22, K2_22, K3_22 and M22 lack
    using Full = NoPart<0, 0>;
    using Imag1 = NoPart<1u << 1, 0>;
    using Real2 = NoPart<0, 1u << 2>;
    using Imag3 = NoPart<1u << 3, 0>;
    using Real4 = NoPart<0, 1u << 4>;
    T c0a = 0, cgra = 0, cgia = 0;
    typename S::Raw fb{}, fc{};
    if (nz >= 2) {
        s.coef(s.load(0), c0a, cgra, cgia);
        fb = s.load(1);
        fc = s.load(2);
    }
    for (int ii = 0; go && ii <= nz - 2; ii += 2) {
        T c0b, cgrb, cgib, c0c, cgrc, cgic;
        s.coef(fb, c0b, cgrb, cgib);
        s.coef(fc, c0c, cgrc, cgic);
        if (ii + 4 <= nz) {
            fb = s.load(ii + 3);
            fc = s.load(ii + 4);
        }
        // T1 = I + dz A_a
        const T ca = dz * c0a, gar = dz * cgra, gai = dz * cgia;
        CPoly<0, T> T11{{{one, ca}}}, T12{{{-gai, gar}}}, T21{{{gai, gar}}};
        CPoly<1, T> T22{{{one, ca}, {T(0), half}}};
        // K2 = dz A_b T1, T2 = I + K2
        CPoly<0, T> K2_11; CPoly<1, T> K2_21, K2_12; CPoly<2, T> K2_22;
        rk_col<Full>(dz * c0b, dz * cgrb, dz * cgib, half, T11, T21, K2_11, K2_21);
        rk_col<Imag1>(dz * c0b, dz * cgrb, dz * cgib, half, T12, T22, K2_12, K2_22);
        CPoly<0, T> U11 = K2_11; CPoly<1, T> U21 = K2_21, U12 = K2_12; CPoly<2, T> U22 = K2_22;
        U11.c[0].r += one;
        U22.c[0].r += one;
        // K3 = 2 dz A_b T2, T3 = I + K3
        CPoly<1, T> K3_11; CPoly<2, T> K3_21, K3_12; CPoly<3, T> K3_22;
        rk_col<Full>(dz2 * c0b, dz2 * cgrb, dz2 * cgib, one, U11, U21, K3_11, K3_21);
        rk_col<Real2>(dz2 * c0b, dz2 * cgrb, dz2 * cgib, one, U12, U22, K3_12, K3_22);
        CPoly<1, T> V11 = K3_11; CPoly<2, T> V21 = K3_21, V12 = K3_12; CPoly<3, T> V22 = K3_22;
        V11.c[0].r += one;
        V22.c[0].r += one;
        // K4/6 = (dz/3) A_c T3: the last term of M, which it starts
        CPoly<2, T> M11; CPoly<3, T> M21, M12; CPoly<4, T> M22;
        rk_col<Full>(dz6 * c0c, dz6 * cgrc, dz6 * cgic, sixth, V11, V21, M11, M21);
        rk_col<Imag3>(dz6 * c0c, dz6 * cgrc, dz6 * cgic, sixth, V12, V22, M12, M22);
        // + K3/3 + (2/3) K2 + Q1/3 + I
        poly_axpy(M11, third, K3_11); poly_axpy(M21, third, K3_21);
        poly_axpy(M12, third, K3_12); poly_axpy<Imag3>(M22, third, K3_22);
        poly_axpy(M11, two3, K2_11); poly_axpy(M21, two3, K2_21);
        poly_axpy(M12, two3, K2_12); poly_axpy<Real2>(M22, two3, K2_22);
        M11.c[0].r += one;
        M11.c[0].i = fm(ca, third, M11.c[0].i);
        M12.c[0].r = fm(-gai, third, M12.c[0].r);
        M12.c[0].i = fm(gar, third, M12.c[0].i);
        M21.c[0].r = fm(gai, third, M21.c[0].r);
        M21.c[0].i = fm(gar, third, M21.c[0].i);
        M22.c[0].r += one;
        M22.c[0].i = fm(ca, third, M22.c[0].i);
        M22.c[1].i += sixth;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const T al = al_[p];
            const cplx<T> m11 = horner(M11, al), m12 = horner(M12, al), m21 = horner(M21, al), m22 = horner<Real4>(M22, al);
            const T y0r = p0r[p], y0i = p0i[p], ygr = pgr[p], ygi = pgi[p];
            p0r[p] = fm(m11.r, y0r, fm(-m11.i, y0i, fm(m12.r, ygr, -m12.i * ygi)));
            p0i[p] = fm(m11.r, y0i, fm(m11.i, y0r, fm(m12.r, ygi, m12.i * ygr)));
            pgr[p] = fm(m21.r, y0r, fm(-m21.i, y0i, fm(m22.r, ygr, -m22.i * ygi)));
            pgi[p] = fm(m21.r, y0i, fm(m21.i, y0r, fm(m22.r, ygi, m22.i * ygr)));
        }
        c0a = c0c; cgra = cgrc; cgia = cgic;
        if constexpr (RS) {
            if (--left == 0) {
                left = every;
                rescale<NP>(p0r, p0i, pgr, pgi);
            }
        }
    }
}

// Largest workgroup of an instance: what its registers leave room for.
constexpr int int_threads(int np) { return np <= 2 ? 1024 : np <= 4 ? 512 : 256; }

// FAST integration: one lane per pixel column and NP precession points, marched
// stage by stage or (POLY) through the shared step matrix.  A column's points,
// and those of several fields (the aperture points of one voxel pass), are
// split over P.nsplit waves of its workgroup, P.split per field; the waves'
// sums are scaled and added to the image in order.  One wave of the split
// gives the bits of a launch of its own that adds to the image.
//
// Bound: one point, HBM; more, the FP32 vector units, and how evenly the waves
// fill them: a wave alone on its SIMD issues an operation every 4.5 cycles,
// several together one every 2.6, and 400 x 400 columns are 2500 waves for
// 1024 SIMDs.  Splitting a column's points over waves evens the load, and
// gives small images parallelism.
template <int NP, bool DENS, bool POLY, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? int_threads(NP) : 256) void k_integrate_fast(FastIntParams P,
                                                                                const void* __restrict__ field,
                                                                                double* __restrict__ img,
                                                                                int accumulate, double inv_total)
{
    const bool go = !P.N.over();                     // (looked at once the first samples are on their way)
    const int64_t plane = (int64_t)P.Mx * P.My;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ns = SPLIT ? P.nsplit : 1, cg = SPLIT ? wave / ns : wave, sp = SPLIT ? wave - cg * ns : 0;
    const int ncg = (int)(blockDim.x >> 6) / ns;
    const int64_t col = ((int64_t)blockIdx.x * ncg + cg) * 64 + lane;
    const bool live = col < plane;
    if (!SPLIT && !live) return;
    const int fld = SPLIT ? sp / P.split : 0, p0 = SPLIT ? (sp - fld * P.split) * NP : 0, at = fld * P.np + p0;
    const FastColumn<DENS, !SPLIT && !POLY> s{field, (live ? col : plane - 1) + fld * P.stride, plane, P.Mz, P.b0, P.bg};
    float p0r[NP], p0i[NP], pgr[NP], pgi[NP];
    if constexpr (POLY) march_poly<NP>(s, P.Mz, P.dz, P.al + at, p0r, p0i, pgr, pgi, go);
    else march_stage<NP>(s, P.Mz, P.dz, P.aa + at, p0r, p0i, pgr, pgi, go);
    double acc = intensity_sum<NP>(min(NP, P.np - p0), p0r, p0i, pgr, pgi) * inv_total;
    if constexpr (SPLIT) {
        __shared__ double part[int_threads(NP)];
        part[threadIdx.x] = acc;
        __syncthreads();
        if (sp > 0 || !live) return;
        for (int k = 0; k < ns; k++) {
            const double v = part[threadIdx.x + 64 * k];
            acc = k > 0 ? acc + v : accumulate ? img[col] + v : v;
        }
        img[col] = acc;
    } else {
        img[col] = accumulate ? img[col] + acc : acc;
    }
}

// ------------------------------------------------------------------ (c) integrate, FP64

struct IntParams {
    int Mx, My, Mz, np;         // np: precession points in this launch
    int nsplit;                 // waves per column
    PointCount N;               // a field of no condition if over
    double b0, bg, dz;
    double aa[INT_SLOTS];       // 2 pi s_g per precession point
    double al[INT_SLOTS];       // 2 dz aa
    int every;                  // double steps between rescalings (0: none)
    int accumulate;             // add the column's sum to img
    double div;                 // and divide by it (0: not yet)
};

// A pixel column of the FP64 field (planes re, im and, DENS, rho).
template <bool DENS>
struct Fp64Column {
    struct Raw {
        double re, im, rho;
    };
    const double *re, *im, *rho;
    int64_t col, plane;
    int nz;
    double b0, bg;
    __device__ __forceinline__ Raw load(int k) const
    {
        const int64_t o = col + plane * (k == nz ? 0 : k);
        Raw v;
        v.re = __builtin_nontemporal_load(re + o);
        v.im = __builtin_nontemporal_load(im + o);
        v.rho = DENS ? __builtin_nontemporal_load(rho + o) : 1.0;
        return v;
    }
    __device__ __forceinline__ void coef(const Raw& f, double& c0, double& cgr, double& cgi) const
    {
        c0 = DENS ? b0 * f.rho : b0;
        const double g = DENS ? bg * f.rho : bg;
        cgr = g * f.re;
        cgi = g * f.im;
    }
};

// Largest workgroup of an instance: what its registers leave room for.
constexpr int int_threads64(int np) { return np <= 3 ? 1024 : np <= 8 ? 512 : 256; }

// dynamicalTwoBeamIntegrationColumn_phaserho (Lib_DynamicalTwoBeamImaging.f90:
// 2316-2480) and the precession average (:1897-1900, 1951): one lane per pixel
// column and NP points, stage by stage or, from six points on, through the
// shared step matrix (40 FMAs per point instead of 80 after ~230 to form the
// matrix: 5 points as 4 + 1 passes take 0.30 ms at 400 x 360 columns of 200
// samples, 6 through the matrix 0.31); a column's points split over P.nsplit
// waves as k_integrate_fast's are; renormalised once at the
// end, as the FAST march is, and (RS) rescaled by powers of two on the way where
// the amplitudes might leave FP64's range.  Bound: FP64 VALU from two points on, HBM below
// (1 point 0.079 ms, 5.8 TB/s).  A march per point with the reference's
// divisions and a square root per step took 0.26 ms for 1 point, 2.00 for 8
// and 8.7 for 32; this takes 0.079, 0.35 and 1.21.
template <int NP, bool DENS, bool SPLIT, bool RS>
__global__ __launch_bounds__(SPLIT ? int_threads64(NP) : 256) void k_integrate_fp64(IntParams P,
                                                                                  const double* __restrict__ fre,
                                                                                  const double* __restrict__ fim,
                                                                                  const double* __restrict__ frho,
                                                                                  double* __restrict__ img)
{
    const bool go = !P.N.over();                     // (looked at once the first samples are on their way)
    const int64_t plane = (int64_t)P.Mx * P.My;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ns = SPLIT ? P.nsplit : 1, cg = SPLIT ? wave / ns : wave, sp = SPLIT ? wave - cg * ns : 0;
    const int ncg = (int)(blockDim.x >> 6) / ns;
    const int64_t col = ((int64_t)blockIdx.x * ncg + cg) * 64 + lane;
    const bool live = col < plane;
    if (!SPLIT && !live) return;
    const Fp64Column<DENS> s{fre, fim, frho, live ? col : plane - 1, plane, P.Mz, P.b0, P.bg};
    const int p0 = sp * NP;
    double p0r[NP], p0i[NP], pgr[NP], pgi[NP];
    if constexpr (NP >= 6) march_poly<NP, RS>(s, P.Mz, P.dz, P.al + p0, p0r, p0i, pgr, pgi, go, P.every);
    else march_stage<NP, RS>(s, P.Mz, P.dz, P.aa + p0, p0r, p0i, pgr, pgi, go, P.every);
    double acc = intensity_sum<NP>(min(NP, P.np - p0), p0r, p0i, pgr, pgi);
    if constexpr (SPLIT) {
        __shared__ double part[int_threads64(NP)];
        part[threadIdx.x] = acc;
        __syncthreads();
        if (sp > 0 || !live) return;
        for (int k = 1; k < ns; k++) acc += part[threadIdx.x + 64 * k];
    }
    if (P.accumulate) acc = img[col] + acc;
    img[col] = P.div != 0.0 ? acc / P.div : acc;
}

}  // namespace d2bi
