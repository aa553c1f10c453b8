// sun_update.hpp -- single-link Cabibbo-Marinari updates (host + device).
//
// heatbath_link restates heatBathSUN (device_PHB_OVR.h:361-485) and overrelax_link
// restates overrelaxationSUN (device_PHB_OVR.h:493-608): N=3 uses the reference's
// block-projection fast path, other N the M = U*F path.  The link, the staple and
// the SU(2) algebra run in the storage precision R; the sampler runs in double for
// FP64 links and in FP32 (generate_su2_milc_f32) for FP32 links.
#pragma once

#include <type_traits>
#include <utility>

#include "sun_rng.hpp"

namespace sun {

template <typename R>
struct Quat {
    R a[4];
};

// v * u^dagger (msu2.h:211-219)
template <typename R>
SUN_HD Quat<R> mul_uv_dagger(const Quat<R>& v, const Quat<R>& u) {
    Quat<R> b;
    b.a[0] = v.a[0] * u.a[0] + v.a[1] * u.a[1] + v.a[2] * u.a[2] + v.a[3] * u.a[3];
    b.a[1] = v.a[1] * u.a[0] - v.a[0] * u.a[1] + v.a[2] * u.a[3] - v.a[3] * u.a[2];
    b.a[2] = v.a[2] * u.a[0] - v.a[0] * u.a[2] + v.a[3] * u.a[1] - v.a[1] * u.a[3];
    b.a[3] = v.a[3] * u.a[0] - v.a[0] * u.a[3] + v.a[1] * u.a[2] - v.a[2] * u.a[1];
    return b;
}

template <typename R>
SUN_HD R qabs(const Quat<R>& r) {
    return sqrt(r.a[0] * r.a[0] + r.a[1] * r.a[1] + r.a[2] * r.a[2] + r.a[3] * r.a[3]);
}

// msu2.h:148-155 (FP32: the reciprocal square root is one v_rsq_f32)
template <typename R>
SUN_HD void conj_normalize(Quat<R>& r) {
    R norm;
    if constexpr (std::is_same<R, float>::value)
        norm = f32_rsq(r.a[0] * r.a[0] + r.a[1] * r.a[1] + r.a[2] * r.a[2] + r.a[3] * r.a[3]);
    else
        norm = R(1) / sqrt(r.a[0] * r.a[0] + r.a[1] * r.a[1] + r.a[2] * r.a[2] + r.a[3] * r.a[3]);
    r.a[0] *= norm;
    r.a[1] *= -norm;
    r.a[2] *= -norm;
    r.a[3] *= -norm;
}

// r r for a unit quaternion in the SU(2) product of msu2.h:90-97:
// (a0^2 - |a|^2, 2 a0 a1, 2 a0 a2, 2 a0 a3)
template <typename R>
SUN_HD Quat<R> quat_square(const Quat<R>& v) {
    Quat<R> r;
    r.a[0] = v.a[0] * v.a[0] - v.a[1] * v.a[1] - v.a[2] * v.a[2] - v.a[3] * v.a[3];
    r.a[1] = R(2) * v.a[0] * v.a[1];
    r.a[2] = R(2) * v.a[0] * v.a[2];
    r.a[3] = R(2) * v.a[0] * v.a[3];
    return r;
}

// rows p,q of U times columns p,q of F, projected on SU(2) (device_PHB_OVR.h:385-400)
template <typename R, int N>
SUN_HD Quat<R> block_projection(const Mat<R, N>& U, const Mat<R, N>& F, int p, int q) {
    cplx<R> a0 = mk<R>(0, 0), a1 = mk<R>(0, 0), a2 = mk<R>(0, 0), a3 = mk<R>(0, 0);
#pragma unroll
    for (int j = 0; j < N; j++) {
        a0 = a0 + U.e[p][j] * F.e[j][p];
        a1 = a1 + U.e[p][j] * F.e[j][q];
        a2 = a2 + U.e[q][j] * F.e[j][p];
        a3 = a3 + U.e[q][j] * F.e[j][q];
    }
    Quat<R> r;
    r.a[0] = a0.re + a3.re;
    r.a[1] = a1.im + a2.im;
    r.a[2] = a1.re - a2.re;
    r.a[3] = a0.im - a3.im;
    return r;
}

// device_PHB_OVR.h:265-272
template <typename R, int N>
SUN_HD Quat<R> get_block_su2(const Mat<R, N>& m, int x, int y) {
    Quat<R> r;
    r.a[0] = m.e[x][x].re + m.e[y][y].re;
    r.a[1] = m.e[x][y].im + m.e[y][x].im;
    r.a[2] = m.e[x][y].re - m.e[y][x].re;
    r.a[3] = m.e[x][x].im - m.e[y][y].im;
    return r;
}

// link <- u * link on rows (x,y) (device_PHB_OVR.h:296-303)
template <typename R, int N>
SUN_HD void mul_block(const Quat<R>& u, Mat<R, N>& link, int x, int y) {
    cplx<R> a00 = mk<R>(u.a[0], u.a[3]), a01 = mk<R>(u.a[2], u.a[1]);
    cplx<R> a10 = mk<R>(-u.a[2], u.a[1]), a11 = mk<R>(u.a[0], -u.a[3]);
#pragma unroll
    for (int j = 0; j < N; j++) {
        cplx<R> tmp = a00 * link.e[x][j] + a01 * link.e[y][j];
        link.e[y][j] = a10 * link.e[x][j] + a11 * link.e[y][j];
        link.e[x][j] = tmp;
    }
}

// one SU(2)-subgroup heatbath step of the N != 3 path on rows (x, y) of block B:
// U <- r U, M <- r M with r = a (M-block)^+ normalised (device_PHB_OVR.h:430-482)
template <typename R, int N, int B, typename DRAWS>
SUN_HD void heatbath_block(Mat<R, N>& U, Mat<R, N>& M, double beta_over_nc, const DrawKey& key, const DRAWS& draws) {
    constexpr int x = block_p(N, B), y = block_q(N, B);
    Quat<R> r = get_block_su2<R, N>(M, x, y);
    R k = qabs(r);
    R ap = R(beta_over_nc) * k;
    k = R(1) / k;
#pragma unroll
    for (int i = 0; i < 4; i++) r.a[i] *= k;
    Quat<R> a;
    const auto bd = draws(B);
    if constexpr (std::is_same<R, float>::value) {
        // FP32 links: the FP32 sampler (as the SU(3) FP32 path)
        generate_su2_milc_f32(ap, key, B, bd.bd, a.a);
    } else {
        double ad[4];
        generate_su2_milc((double)ap, key, B, bd, ad);
#pragma unroll
        for (int i = 0; i < 4; i++) a.a[i] = R(ad[i]);
    }
    const Quat<R> rr = mul_uv_dagger(a, r);
    mul_block<R, N>(rr, U, x, y);
    mul_block<R, N>(rr, M, x, y);
}

template <typename R, int N, typename DRAWS, int... B>
SUN_HD void heatbath_blocks(Mat<R, N>& U, Mat<R, N>& M, double beta_over_nc, const DrawKey& key, const DRAWS& draws,
                            std::integer_sequence<int, B...>) {
    (heatbath_block<R, N, B>(U, M, beta_over_nc, key, draws), ...);
}

// draws(block): the draws of a subgroup (KeyDraws, or the same computed before)
template <typename R, int N, typename DRAWS>
SUN_HD void heatbath_link(Mat<R, N>& U, const Mat<R, N>& F, double beta_over_nc, const DrawKey& key,
                          const DRAWS& draws) {
    if constexpr (N == 3) {
#pragma unroll
        for (int block = 0; block < 3; block++) {
            const int p = block_p(3, block), q = block_q(3, block);
            Quat<R> r = block_projection<R, 3>(U, F, p, q);
            R k = qabs(r);
            R ap = R(beta_over_nc) * k;
            k = R(1) / k;
#pragma unroll
            for (int i = 0; i < 4; i++) r.a[i] *= k;
            double ad[4];
            generate_su2_milc((double)ap, key, block, draws(block), ad);
            Quat<R> a;
#pragma unroll
            for (int i = 0; i < 4; i++) a.a[i] = R(ad[i]);
            r = mul_uv_dagger(a, r);
            cplx<R> b0 = mk<R>(r.a[0], r.a[3]), b1 = mk<R>(r.a[2], r.a[1]);
            cplx<R> b2 = mk<R>(-r.a[2], r.a[1]), b3 = mk<R>(r.a[0], -r.a[3]);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                cplx<R> tmp0 = b0 * U.e[p][j] + b1 * U.e[q][j];
                U.e[q][j] = b2 * U.e[p][j] + b3 * U.e[q][j];
                U.e[p][j] = tmp0;
            }
        }
    } else {
        Mat<R, N> M = U * F;
        // one instance per block: the block's rows are compile-time constants (a
        // rolled loop would index U and M at run time, i.e. from scratch memory)
        heatbath_blocks<R, N>(U, M, beta_over_nc, key, draws, std::make_integer_sequence<int, N * (N - 1) / 2>{});
    }
}

template <typename R, int N>
SUN_HD void heatbath_link(Mat<R, N>& U, const Mat<R, N>& F, double beta_over_nc, const DrawKey& key) {
    heatbath_link<R, N>(U, F, beta_over_nc, key, [&](int block) { return KeyDraws(key, block); });
}

template <typename R, int N>
SUN_HD void overrelax_link(Mat<R, N>& U, const Mat<R, N>& F) {
    if constexpr (N == 3) {
#pragma unroll
        for (int block = 0; block < 3; block++) {
            const int p = block_p(3, block), q = block_q(3, block);
            Quat<R> r = block_projection<R, 3>(U, F, p, q);
            conj_normalize(r);
            cplx<R> b0 = mk<R>(r.a[0], r.a[3]), b1 = mk<R>(r.a[2], r.a[1]);
            cplx<R> b2 = mk<R>(-r.a[2], r.a[1]), b3 = mk<R>(r.a[0], -r.a[3]);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                cplx<R> tmp0 = b0 * U.e[p][j] + b1 * U.e[q][j];
                cplx<R> tmp1 = b2 * U.e[p][j] + b3 * U.e[q][j];
                U.e[p][j] = b0 * tmp0 + b1 * tmp1;
                U.e[q][j] = b2 * tmp0 + b3 * tmp1;
            }
        }
    } else {
        Mat<R, N> M = U * F;
#pragma unroll
        for (int block = 0; block < N * (N - 1) / 2; block++) {
            const int x = block_p(N, block), y = block_q(N, block);
            Quat<R> r = get_block_su2<R, N>(M, x, y);
            conj_normalize(r);
            if constexpr (std::is_same<R, float>::value) {
                // FP32 links: the rotation applied once as r^2 (half the row updates;
                // equal to applying r twice up to FP32 rounding)
                const Quat<R> r2 = quat_square(r);
                mul_block<R, N>(r2, U, x, y);
                mul_block<R, N>(r2, M, x, y);
            } else {
                mul_block<R, N>(r, U, x, y);
                mul_block<R, N>(r, U, x, y);
                mul_block<R, N>(r, M, x, y);
                mul_block<R, N>(r, M, x, y);
            }
        }
    }
}

// Projection onto SU(N) by SU(2)-subgroup maximisation of Re Tr(w q^+)
// (projectlink.h:16-64, project_link): per hit, for every subgroup block, the block
// of w q^+ is normalised, conjugated and multiplied into w from the left.  With
// tol > 0 the hits stop once the relative change of Re Tr(w q) / N (the reference's
// measure, realtraceUVdagger of w and the daggered q) falls to tol.  SU3project
// (projectlink.h:119-139), the reference's N = 3 choice, is this with w = 1,
// tol = 0 and the blocks (0,1), (1,2), (0,2); it has no zero-block guard (a block
// of exactly zero norm would give NaN there and the identity block here).
// In FP32 with a tolerance the stop is decided by the rounding of the trace (1e-7 against
// tolerances of 1e-10), so every rounding counts: project_link_rounded keeps the separately
// rounded steps.
template <typename R, int N>
SUN_HD R retrace_rounded(const Mat<R, N>& a, const Mat<R, N>& b) {  // Re Tr(a b) with b stored daggered
    R s = R(0);
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j < N; j++) s += a.e[i][j].re * b.e[i][j].re + a.e[i][j].im * b.e[i][j].im;
    return s;
}

template <typename R, int N>
SUN_HD void project_link_rounded(Mat<R, N>& w, const Mat<R, N>& q_in, int nhit, R tol) {
    const Mat<R, N> q = dagger(q_in);
    R conver = R(1), old_tr = R(0);
    if (tol > R(0)) old_tr = retrace_rounded<R, N>(w, q) / R(N);
#pragma unroll 1
    for (int hit = 0; hit < nhit && conver > tol; hit++) {
        // unrolled: compile-time rows keep w in registers
#pragma unroll
        for (int block = 0; block < N * (N - 1) / 2; block++) {
            const int x = block_p(N, block), y = block_q(N, block);
            const Mat<R, N> action = w * q;
            Quat<R> r = get_block_su2<R, N>(action, x, y);
            R k = qabs(r);
            if (k == R(0)) {
                k = R(1);
                r.a[0] = R(1);
            }
            k = R(1) / k;
            r.a[0] *= k;
            r.a[1] *= -k;
            r.a[2] *= -k;
            r.a[3] *= -k;
            mul_block<R, N>(r, w, x, y);
        }
        if (tol > R(0)) {
            const R new_tr = retrace_rounded<R, N>(w, q) / R(N);
            conver = (new_tr - old_tr) / old_tr;
            old_tr = new_tr;
        }
    }
}

// Otherwise fused multiply-adds throughout, and 1/|r| by the hardware's reciprocal square root
// (FP64 with a correction step to full precision, FP32 with one of the rotation).  The hits are a
// serial chain of arithmetic that bounds the smearing kernels: 3 x ~105 instructions per SU(3)
// hit, half of the separately rounded form with its square root and division.
template <typename R, int N>
SUN_HD R retrace_conj(const Mat<R, N>& a, const Mat<R, N>& b) {  // Re Tr(a b) with b stored daggered
    R s = R(0);
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j < N; j++) s = fma(a.e[i][j].im, b.e[i][j].im, fma(a.e[i][j].re, b.e[i][j].re, s));
    return s;
}

SUN_HD double inv_sqrt(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    if (x > 1e-290 && x < 1e290) {
        const double y = __builtin_amdgcn_rsq(x), e = fma(-x * y, y, 1.0);
        return fma(y * e, fma(0.375, e, 0.5), y);
    }
#endif
    return 1.0 / sqrt(x);
}
SUN_HD float inv_sqrt(float x) {
    if (x < 1e-30f) return 1e15f * f32_rsq(x * 1e30f);  // the native instruction flushes denormals
    return f32_rsq(x);
}

// A rotation that is unitary but for rounding, scaled to |r| = 1.  FP32: what the reciprocal root
// leaves (1e-7, leaning to -7e-9), and what rounding does next to r0 = 1, where the numbers
// below lie twice as close as those above.  Mean |U|^2 / N - 1 after ten hits, SU(3) and SU(4):
// -3.5e-7 and -4.9e-7 without, -9e-8 and -1e-7 with square roots and divisions, 5e-9 and 1e-8
// so (one APE direction of 24^3 x 32 SU(3) 12-real 61.5 -> 63 us, SU(4) 16^3 x 32 50.6 -> 52).
SUN_HD void unit(Quat<float>& r) {
    float s = fmaf(-r.a[0], r.a[0], 1.f);
    s = fmaf(-r.a[1], r.a[1], s);
    s = fmaf(-r.a[2], r.a[2], s);
    s = 0.5f * fmaf(-r.a[3], r.a[3], s);
#pragma unroll
    for (int i = 0; i < 4; i++) r.a[i] = fmaf(s, r.a[i], r.a[i]);
}
SUN_HD void unit(Quat<double>&) {}  // inv_sqrt is good to the last bit

// 2 Re and Im combinations of the (x, y) block of w q (get_block_su2 of the product)
template <typename R, int N>
SUN_HD Quat<R> product_block(const Mat<R, N>& w, const Mat<R, N>& q, int x, int y) {
    R r0 = R(0), r1 = R(0), r2 = R(0), r3 = R(0);
#pragma unroll
    for (int k = 0; k < N; k++) {
        const cplx<R> a = w.e[x][k], b = w.e[y][k], c = q.e[k][x], d = q.e[k][y];
        r0 = fma(-b.im, d.im, fma(b.re, d.re, fma(-a.im, c.im, fma(a.re, c.re, r0))));
        r1 = fma(b.im, c.re, fma(b.re, c.im, fma(a.im, d.re, fma(a.re, d.im, r1))));
        r2 = fma(b.im, c.im, fma(-b.re, c.re, fma(-a.im, d.im, fma(a.re, d.re, r2))));
        r3 = fma(-b.im, d.re, fma(-b.re, d.im, fma(a.im, c.re, fma(a.re, c.im, r3))));
    }
    return Quat<R>{{r0, r1, r2, r3}};
}

// rows x, y of w <- u times them (mul_block)
template <typename R, int N>
SUN_HD void rotate_rows(const Quat<R>& u, Mat<R, N>& w, int x, int y) {
    const R u0 = u.a[0], u1 = u.a[1], u2 = u.a[2], u3 = u.a[3];
#pragma unroll
    for (int j = 0; j < N; j++) {
        const cplx<R> a = w.e[x][j], b = w.e[y][j];
        w.e[x][j] = mk<R>(fma(-u1, b.im, fma(u2, b.re, fma(-u3, a.im, u0 * a.re))),
                          fma(u1, b.re, fma(u2, b.im, fma(u3, a.re, u0 * a.im))));
        w.e[y][j] = mk<R>(fma(u3, b.im, fma(u0, b.re, fma(-u1, a.im, -u2 * a.re))),
                          fma(-u3, b.re, fma(u0, b.im, fma(u1, a.re, -u2 * a.im))));
    }
}

template <typename R, int N>
SUN_HD void project_link(Mat<R, N>& w, const Mat<R, N>& q_in, int nhit, R tol) {
    if constexpr (sizeof(R) == 4) {
        if (tol > R(0)) {
            project_link_rounded<R, N>(w, q_in, nhit, tol);
            return;
        }
    }
    const Mat<R, N> q = dagger(q_in);
    R conver = R(1), old_tr = R(0);
    if (tol > R(0)) old_tr = retrace_conj<R, N>(w, q) / R(N);
#pragma unroll 1
    for (int hit = 0; hit < nhit && conver > tol; hit++) {
        // unrolled: compile-time rows keep w in registers
#pragma unroll
        for (int block = 0; block < N * (N - 1) / 2; block++) {
            const int x = block_p(N, block), y = block_q(N, block);
            Quat<R> r = product_block<R, N>(w, q, x, y);
            const R n2 = fma(r.a[3], r.a[3], fma(r.a[2], r.a[2], fma(r.a[1], r.a[1], r.a[0] * r.a[0])));
            if (n2 == R(0)) {
                r.a[0] = R(1);
            } else {
                const R k = inv_sqrt(n2);
                r.a[0] *= k;
                r.a[1] *= -k;
                r.a[2] *= -k;
                r.a[3] *= -k;
                unit(r);
            }
            rotate_rows<R, N>(r, w, x, y);
        }
        if (tol > R(0)) {
            const R new_tr = retrace_conj<R, N>(w, q) / R(N);
            conver = (new_tr - old_tr) / old_tr;
            old_tr = new_tr;
        }
    }
}

// Reunitarisation (reunitlink.h:16-85).  N=3: row Gram-Schmidt + cross product;
// N>3: column Gram-Schmidt + determinant phase on the last column.  N=2 is not
// compilable in the reference (reunitlink.h:86); here the textbook projection
// a=(U00+conj U11)/2, b=(U01-conj U10)/2, normalised.
template <typename R, int N>
SUN_HD void reunit_link(Mat<R, N>& U) {
    if constexpr (N == 3) {
        R t1 = R(0);
        cplx<R> t2 = mk<R>(0, 0);
#pragma unroll
        for (int c = 0; c < 3; c++) t1 += abs2(U.e[0][c]);
        t1 = R(1) / sqrt(t1);
#pragma unroll
        for (int c = 0; c < 3; c++) U.e[0][c] = scale(U.e[0][c], t1);
#pragma unroll
        for (int c = 0; c < 3; c++) t2 = t2 + conj(U.e[0][c]) * U.e[1][c];
#pragma unroll
        for (int c = 0; c < 3; c++) U.e[1][c] = U.e[1][c] - t2 * U.e[0][c];
        t1 = R(0);
#pragma unroll
        for (int c = 0; c < 3; c++) t1 += abs2(U.e[1][c]);
        t1 = R(1) / sqrt(t1);
#pragma unroll
        for (int c = 0; c < 3; c++) U.e[1][c] = scale(U.e[1][c], t1);
        reconstruct_row2(U);
    } else if constexpr (N == 2) {
        cplx<R> a = mk<R>((U.e[0][0].re + U.e[1][1].re) * R(0.5), (U.e[0][0].im - U.e[1][1].im) * R(0.5));
        cplx<R> b = mk<R>((U.e[0][1].re - U.e[1][0].re) * R(0.5), (U.e[0][1].im + U.e[1][0].im) * R(0.5));
        R n = R(1) / sqrt(abs2(a) + abs2(b));
        a = scale(a, n);
        b = scale(b, n);
        U.e[0][0] = a;
        U.e[0][1] = b;
        U.e[1][0] = mk<R>(-b.re, b.im);
        U.e[1][1] = conj(a);
    } else {
        R t1 = R(0);
        cplx<R> t2;
#pragma unroll
        for (int c = 0; c < N; c++) t1 += abs2(U.e[c][0]);
        t1 = R(1) / sqrt(t1);
#pragma unroll
        for (int c = 0; c < N; c++) U.e[c][0] = scale(U.e[c][0], t1);
#pragma unroll
        for (int j = 1; j < N; j++) {
#pragma unroll
            for (int i = 0; i < j; i++) {
                t2 = conj(U.e[0][i]) * U.e[0][j];
#pragma unroll
                for (int c = 1; c < N; ++c) t2 = t2 + conj(U.e[c][i]) * U.e[c][j];
#pragma unroll
                for (int c = 0; c < N; ++c) U.e[c][j] = U.e[c][j] - t2 * U.e[c][i];
            }
            t1 = R(0);
#pragma unroll
            for (int c = 0; c < N; ++c) t1 += abs2(U.e[c][j]);
            t1 = R(1) / sqrt(t1);
#pragma unroll
            for (int c = 0; c < N; ++c) U.e[c][j] = scale(U.e[c][j], t1);
        }
        t2 = det<R, N>(U);
        const R ai = arg_of(t2);
        R sn, cs;
        sincos_of(ai, sn, cs);
        t2 = mk<R>(cs, -sn);
#pragma unroll
        for (int c = 0; c < N; ++c) U.e[c][N - 1] = U.e[c][N - 1] * t2;
    }
}


// exp(iQ) for a traceless Hermitian 3x3 Q (Morningstar and Peardon, Phys. Rev. D 69
// (2004) 054501, eqs. (19)-(34)): exp(iQ) = f0 + f1 Q + f2 Q^2 with the f_j from
// c0 = det Q = Tr Q^3 / 3 and c1 = Tr Q^2 / 2.  For c1 below kStoutSeriesC1 (|Q| <
// 0.08) the f_j are the exponential series reduced by Cayley-Hamilton,
// Q^3 = c1 Q + c0, summed to order 16 (the closed form divides by ~c1 there).
constexpr double kStoutSeriesC1 = 4.0e-3;

SUN_HD void exp_iq_su3(const Mat<double, 3>& Q, Mat<double, 3>& E) {
    const Mat<double, 3> QQ = Q * Q;
    const double c1 = 0.5 * realtrace(QQ);
    const double c0 = realtrace(Q * QQ) / 3.0;
    cplx<double> f0, f1, f2;
    if (c1 < kStoutSeriesC1) {
        // Q^k = a + b Q + c Q^2 -> Q^(k+1) = c c0 + (a + c c1) Q + b Q^2
        double a = 1.0, b = 0.0, c = 0.0;
        cplx<double> t = mk<double>(1.0, 0.0);  // i^k / k!
        f0 = f1 = f2 = mk<double>(0.0, 0.0);
#pragma unroll 1
        for (int k = 0; k <= 16; k++) {
            f0 = f0 + scale(t, a);
            f1 = f1 + scale(t, b);
            f2 = f2 + scale(t, c);
            const double na = c * c0, nb = a + c * c1, nc = b;
            a = na;
            b = nb;
            c = nc;
            t = mk<double>(-t.im / (k + 1), t.re / (k + 1));
        }
    } else {
        const double c0abs = fabs(c0);
        const double s3 = sqrt(c1 / 3.0);
        const double c0max = 2.0 * (c1 / 3.0) * s3;
        const double theta = acos(fmin(c0abs / c0max, 1.0));
        const double u = s3 * cos(theta / 3.0), w = sqrt(c1) * sin(theta / 3.0);
        const double u2 = u * u, w2 = w * w;
        const double xi0 = fabs(w) < 0.05 ? 1.0 - w2 / 6.0 * (1.0 - w2 / 20.0 * (1.0 - w2 / 42.0)) : sin(w) / w;
        const double cw = cos(w);
        const cplx<double> e2iu = mk<double>(cos(2.0 * u), sin(2.0 * u));
        const cplx<double> emiu = mk<double>(cos(u), -sin(u));
        const cplx<double> h0 = scale(e2iu, u2 - w2) + emiu * mk<double>(8.0 * u2 * cw, 2.0 * u * (3.0 * u2 + w2) * xi0);
        const cplx<double> h1 = scale(e2iu, 2.0 * u) - emiu * mk<double>(2.0 * u * cw, -(3.0 * u2 - w2) * xi0);
        const cplx<double> h2 = e2iu - emiu * mk<double>(cw, 3.0 * u * xi0);
        const double den = 1.0 / (9.0 * u2 - w2);
        f0 = scale(h0, den);
        f1 = scale(h1, den);
        f2 = scale(h2, den);
        if (c0 < 0) {  // f_j(-c0) = (-1)^j conj f_j(c0)
            f0 = conj(f0);
            f1 = mk<double>(-f1.re, f1.im);
            f2 = conj(f2);
        }
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cplx<double> e = f1 * Q.e[i][j] + f2 * QQ.e[i][j];
            if (i == j) e = e + f0;
            E.e[i][j] = e;
        }
}

// One stout step of a link (stout.cu:86-92, 519-535): Omega = V U^+ with V = rho x
// the staple sum, Q = the traceless part of (i/2)(Omega^+ - Omega), W = exp(iQ) U.
SUN_HD Mat<double, 3> stout_link(const Mat<double, 3>& V, const Mat<double, 3>& U) {
    const Mat<double, 3> Om = V * dagger(U);
    Mat<double, 3> Q;
    cplx<double> tr = mk<double>(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            // (i/2)(conj(Om_ji) - Om_ij)
            const cplx<double> d = conj(Om.e[j][i]) - Om.e[i][j];
            Q.e[i][j] = mk<double>(-0.5 * d.im, 0.5 * d.re);
        }
#pragma unroll
    for (int i = 0; i < 3; i++) tr = tr + Q.e[i][i];
#pragma unroll
    for (int i = 0; i < 3; i++) Q.e[i][i] = Q.e[i][i] - scale(tr, 1.0 / 3.0);
    Mat<double, 3> E;
    exp_iq_su3(Q, E);
    return E * U;
}

}  // namespace sun
