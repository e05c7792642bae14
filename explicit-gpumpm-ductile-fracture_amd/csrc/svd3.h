// svd3.h — 3x3 singular value decomposition for one particle per lane.
//
// Same algorithm and sign/ordering conventions as the reference's QR/Givens
// SVD (QRSVD.hpp:226-374 with givens.hpp:12-210): Givens upper
// bidiagonalisation, implicit Wilkinson-shift QR sweeps until a diagonal or
// super-diagonal entry drops below 128*eps*max(|B|/2, 1), then a 2x2 polar +
// symmetric eigen step on the remaining block and the reference's sort/sign
// fix-up, so that F = U diag(S) V^T with S0 >= S1 >= |S2| and only S2 < 0.
//
// Written for registers: matrices are plain T[3][3] arrays fully unrolled by
// the compiler; a Givens rotation is (i, k, c, s).  The sweep loop is bounded
// (kMaxSweeps) so that a non-converging input can never stall a wavefront; the
// reference loop is unbounded.  Templated on float and double.  It serves the FP32
// stress arithmetic and its FP64 redo; the default FP64 update takes the principal
// axes below.
#pragma once
#include <hip/hip_runtime.h>

namespace mpmx {

template <typename T> struct Eps;
template <> struct Eps<float>  { static constexpr float  v = 1.1920928955078125e-07f; };
template <> struct Eps<double> { static constexpr double v = 2.220446049250313080847e-16; };

constexpr int kMaxSweeps = 64;

template <typename T>
struct Rot {
    int i, k;
    T c, s;
};

template <typename T>
__device__ __forceinline__ Rot<T> rot_id(int i, int k) { return Rot<T>{i, k, T(1), T(0)}; }

// 1 / sqrt(d) for d > 0.  FP64: the hardware estimate refined by two Newton
// steps, y += y (1 - d y^2) / 2 (within about an ulp of 1/sqrt(d), a tenth of
// the instructions of a square root and a division); FP32: 1 / sqrtf.
__device__ __forceinline__ float rsqrt_acc(float d) { return 1.0f / sqrtf(d); }
__device__ __forceinline__ double rsqrt_acc(double d) {
    double y = __builtin_amdgcn_rsq(d);
    double e = fma(-d * y, y, 1.0);
    y = fma(y * 0.5, e, y);
    e = fma(-d * y, y, 1.0);
    return fma(y * 0.5, e, y);
}

// [c -s; s c] [a; b] = [*; 0]
template <typename T>
__device__ __forceinline__ void rot_conv(Rot<T>& g, T a, T b) {
    const T d = a * a + b * b;
    g.c = T(1); g.s = T(0);
    if (d != T(0)) { const T t = rsqrt_acc(d); g.c = a * t; g.s = -b * t; }
}
// [c -s; s c] [a; b] = [0; *]
template <typename T>
__device__ __forceinline__ void rot_unconv(Rot<T>& g, T a, T b) {
    const T d = a * a + b * b;
    g.c = T(0); g.s = T(1);
    if (d != T(0)) { const T t = rsqrt_acc(d); g.s = a * t; g.c = b * t; }
}
// rows i,k of A
template <typename T, int NC>
__device__ __forceinline__ void rot_rows(const Rot<T>& g, T (&A)[NC][NC]) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const T a = A[g.i][j], b = A[g.k][j];
        A[g.i][j] = g.c * a - g.s * b;
        A[g.k][j] = g.s * a + g.c * b;
    }
}
// columns i,k of A
template <typename T>
__device__ __forceinline__ void rot_cols(const Rot<T>& g, T (&A)[3][3]) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const T a = A[r][g.i], b = A[r][g.k];
        A[r][g.i] = g.c * a - g.s * b;
        A[r][g.k] = g.s * a + g.c * b;
    }
}

template <typename T>
__device__ __forceinline__ void eye3(T (&A)[3][3]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) A[r][c] = (r == c) ? T(1) : T(0);
}

// bring [x x 0; x x x; 0 0 x] to upper bidiagonal, accumulating U and V
template <typename T>
__device__ __forceinline__ void chase(T (&H)[3][3], T (&U)[3][3], T (&V)[3][3]) {
    Rot<T> r1 = rot_id<T>(0, 1);
    rot_conv(r1, H[0][0], H[1][0]);
    Rot<T> r2 = rot_id<T>(1, 2);
    if (H[1][0] != T(0))
        rot_conv(r2, H[0][0] * H[0][1] + H[1][0] * H[1][1], H[0][0] * H[0][2] + H[1][0] * H[1][2]);
    else
        rot_conv(r2, H[0][1], H[0][2]);
    rot_rows(r1, H);
    rot_cols(r2, H);
    rot_cols(r2, V);
    Rot<T> r3 = rot_id<T>(1, 2);
    rot_conv(r3, H[1][1], H[2][1]);
    rot_rows(r3, H);
    rot_cols(r1, U);
    rot_cols(r3, U);
}

// 2x2 block at (t,t): polar rotation, then the symmetric 2x2 eigen rotation
template <typename T>
__device__ __forceinline__ void block2(int t, const T (&B)[3][3], T (&U)[3][3], T (&S)[3], T (&V)[3][3]) {
    const int other = (t == 1) ? 0 : 2;
    S[other] = B[other][other];
    T A2[2][2] = {{B[t][t], B[t][t + 1]}, {B[t + 1][t], B[t + 1][t + 1]}};
    Rot<T> u = rot_id<T>(0, 1), v = rot_id<T>(0, 1);
    // polar part
    const T x0 = A2[0][0] + A2[1][1], x1 = A2[1][0] - A2[0][1];
    const T d2 = x0 * x0 + x1 * x1;
    if (d2 != T(0)) { const T t = rsqrt_acc(d2); u.c = x0 * t; u.s = -x1 * t; }
    rot_rows(u, A2);
    // symmetric part
    const T x = A2[0][0], y = A2[0][1], z = A2[1][1];
    const T y2 = y * y;
    T cs, sn, s0, s1;
    if (y2 == T(0)) {
        cs = T(1); sn = T(0); s0 = x; s1 = z;
    } else {
        const T tau = T(0.5) * (x - z);
        const T w = sqrt(tau * tau + y2);
        const T tt = (tau > T(0)) ? y / (tau + w) : y / (tau - w);
        cs = rsqrt_acc(tt * tt + T(1));
        sn = -tt * cs;
        const T c2 = cs * cs, s2 = sn * sn, csy2 = T(2) * cs * sn * y;
        s0 = c2 * x - csy2 + s2 * z;
        s1 = s2 * x + csy2 + c2 * z;
    }
    if (s0 < s1) { const T tmp = s0; s0 = s1; s1 = tmp; v.c = -sn; v.s = cs; }
    else         { v.c = cs; v.s = sn; }
    // u <- u * v
    const T nc = u.c * v.c - u.s * v.s, ns = u.s * v.c + u.c * v.s;
    u.c = nc; u.s = ns;
    S[t] = s0;
    S[t + 1] = s1;
    u.i += t; u.k += t;
    v.i += t; v.k += t;
    rot_cols(u, U);
    rot_cols(v, V);
}

template <typename T>
__device__ __forceinline__ void swapv(T& a, T& b) { const T t = a; a = b; b = t; }
template <typename T>
__device__ __forceinline__ void swapc(T (&A)[3][3], int a, int b) {
#pragma unroll
    for (int r = 0; r < 3; ++r) swapv(A[r][a], A[r][b]);
}
template <typename T>
__device__ __forceinline__ void negc(T (&A)[3][3], int a) {
#pragma unroll
    for (int r = 0; r < 3; ++r) A[r][a] = -A[r][a];
}
template <typename T>
__device__ __forceinline__ void flip(int j, T (&U)[3][3], T (&S)[3]) {
    S[j] = -S[j];
    negc(U, j);
}

// ordering/sign fix-up after a block at t = 0 (rows/cols 0,1)
template <typename T>
__device__ __forceinline__ void order0(T (&U)[3][3], T (&s)[3], T (&V)[3][3]) {
    if (fabs(s[1]) >= fabs(s[2])) {
        if (s[1] < T(0)) { flip(1, U, s); flip(2, U, s); }
        return;
    }
    if (s[2] < T(0)) { flip(1, U, s); flip(2, U, s); }
    swapv(s[1], s[2]); swapc(U, 1, 2); swapc(V, 1, 2);
    if (s[1] > s[0]) { swapv(s[0], s[1]); swapc(U, 0, 1); swapc(V, 0, 1); }
    else { negc(U, 2); negc(V, 2); }
}
// ordering/sign fix-up after a block at t = 1 (rows/cols 1,2)
template <typename T>
__device__ __forceinline__ void order1(T (&U)[3][3], T (&s)[3], T (&V)[3][3]) {
    if (fabs(s[0]) >= s[1]) {
        if (s[0] < T(0)) { flip(0, U, s); flip(2, U, s); }
        return;
    }
    swapv(s[0], s[1]); swapc(U, 0, 1); swapc(V, 0, 1);
    if (fabs(s[1]) < fabs(s[2])) { swapv(s[1], s[2]); swapc(U, 1, 2); swapc(V, 1, 2); }
    else { negc(U, 1); negc(V, 1); }
    if (s[1] < T(0)) { flip(1, U, s); flip(2, U, s); }
}

// A (row-major 3x3) -> U, S, V with A = U diag(S) V^T.  Returns sweeps used.
template <typename T>
__device__ __forceinline__ int svd3(const T (&A)[3][3], T (&U)[3][3], T (&S)[3], T (&V)[3][3]) {
    T B[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) B[r][c] = A[r][c];
    eye3(U);
    eye3(V);
    {
        Rot<T> r = rot_id<T>(1, 2);
        rot_conv(r, B[1][0], B[2][0]);
        rot_rows(r, B);
        rot_cols(r, U);
        chase(B, U, V);
    }
    T a0 = B[0][0], a1 = B[1][1], a2 = B[2][2], b0 = B[0][1], b1 = B[1][2];
    const T nrm = T(0.5) * sqrt(a0 * a0 + a1 * a1 + a2 * a2 + b0 * b0 + b1 * b1);
    const T tol = Eps<T>::v * T(128) * (nrm > T(1) ? nrm : T(1));
    int sweeps = 0;
    while (fabs(a0) > tol && fabs(a1) > tol && fabs(a2) > tol && fabs(b0) > tol && fabs(b1) > tol &&
           sweeps < kMaxSweeps) {
        // Wilkinson shift of the trailing 2x2 of B^T B
        const T ta = a1 * a1 + b0 * b0, tc = a2 * a2 + b1 * b1, tb = a1 * b1;
        const T dd = T(0.5) * (ta - tc);
        const T bs = tb * tb;
        const T mu = tc - copysign(bs / (fabs(dd) + sqrt(dd * dd + bs)), dd);
        Rot<T> r = rot_id<T>(0, 1);
        rot_conv(r, a0 * a0 - mu, a0 * b0);
        rot_cols(r, B);
        rot_cols(r, V);
        chase(B, U, V);
        a0 = B[0][0]; a1 = B[1][1]; a2 = B[2][2]; b0 = B[0][1]; b1 = B[1][2];
        ++sweeps;
    }
    S[0] = S[1] = S[2] = T(0) / T(0);
    if (fabs(b1) <= tol) {
        block2<T>(0, B, U, S, V);
        order0(U, S, V);
    } else if (fabs(b0) <= tol) {
        block2<T>(1, B, U, S, V);
        order1(U, S, V);
    } else if (fabs(a1) <= tol) {
        Rot<T> r1 = rot_id<T>(1, 2);
        rot_unconv(r1, B[1][2], B[2][2]);
        rot_rows(r1, B);
        rot_cols(r1, U);
        block2<T>(0, B, U, S, V);
        order0(U, S, V);
    } else if (fabs(a2) <= tol) {
        Rot<T> r1 = rot_id<T>(1, 2);
        rot_conv(r1, B[1][1], B[1][2]);
        rot_cols(r1, B);
        rot_cols(r1, V);
        Rot<T> r2 = rot_id<T>(0, 2);
        rot_conv(r2, B[0][0], B[0][2]);
        rot_cols(r2, B);
        rot_cols(r2, V);
        block2<T>(0, B, U, S, V);
        order0(U, S, V);
    } else if (fabs(a0) <= tol) {
        Rot<T> r1 = rot_id<T>(0, 1);
        rot_unconv(r1, B[0][1], B[1][1]);
        rot_rows(r1, B);
        rot_cols(r1, U);
        Rot<T> r2 = rot_id<T>(0, 2);
        rot_unconv(r2, B[0][2], B[2][2]);
        rot_rows(r2, B);
        rot_cols(r2, U);
        block2<T>(1, B, U, S, V);
        order1(U, S, V);
    }
    return sweeps;
}

// ---- principal axes in FP64 ----------------------------------------------------
// The isotropic updates need the left singular vectors and the singular values
// only: functions of them act on F as sum_a f_a u_a u_a^T F, so V is never formed.
// One-sided Jacobi: rotations from the right make the columns of G = F V
// orthogonal; then |g_a| = |S_a| and u_a = g_a / |S_a|.  It works on F itself (a
// product F F^T would square the condition number), needs two reciprocal square
// roots and 27 multiply-adds per rotation, no division, and keeps nine doubles,
// where the QR iteration above keeps B, U and V.  A pair of columns counts as
// orthogonal below 2^-50 of their lengths' product.
constexpr int kMaxJacobi = 32;

__device__ __forceinline__ void jacobi_columns(double (&G)[3][3]) {
    constexpr double tol2 = 0x1p-100;
    for (int sweep = 0; sweep < kMaxJacobi; ++sweep) {
        bool turned = false;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int p = k == 2 ? 1 : 0, q = k == 0 ? 1 : 2;
            const double a = fma(G[2][p], G[2][p], fma(G[1][p], G[1][p], G[0][p] * G[0][p]));
            const double b = fma(G[2][q], G[2][q], fma(G[1][q], G[1][q], G[0][q] * G[0][q]));
            const double c = fma(G[2][p], G[2][q], fma(G[1][p], G[1][q], G[0][p] * G[0][q]));
            // below 2^-48 of the other's length a column is rounding noise (of a
            // matrix of lower rank): more rotations would only take it on to
            // lengths far below that
            const bool noise = abs(__double2hiint(a) - __double2hiint(b)) >= 96 << 20;
            if (c * c > tol2 * (a * b) && !noise) {
                // tan 2t = 2c / (b - a); cos t >= sqrt(1/2)
                const double d = b - a, r = rsqrt_acc(fma(d, d, 4.0 * (c * c)));
                const double h = fma(0.5 * fabs(d), r, 0.5), rh = rsqrt_acc(h);
                const double cs = h * rh, sn = copysign(1.0, d) * (c * r) * rh;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double x = G[i][p], y = G[i][q];
                    G[i][p] = fma(cs, x, -sn * y);
                    G[i][q] = fma(sn, x, cs * y);
                }
                turned = true;
            }
        }
        if (!turned) break;
    }
}

// F = sum_a S_a u_a v_a^T, u_a the columns of U, R_a = 1 / S_a; no order, at most
// one S_a < 0 (the smallest, where det F < 0).  False where the smallest is below
// 1e-5 of the largest: there u_a is not to be had from g_a, nor v_a from u_a^T F.
__device__ __forceinline__ bool principal_axes(const float (&F)[3][3], double (&U)[3][3], double (&S)[3],
                                               double (&R)[3]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) U[r][c] = F[r][c];
    jacobi_columns(U);
    const double det = U[0][0] * (U[1][1] * U[2][2] - U[1][2] * U[2][1]) -
                       U[0][1] * (U[1][0] * U[2][2] - U[1][2] * U[2][0]) +
                       U[0][2] * (U[1][0] * U[2][1] - U[1][1] * U[2][0]);
    double n2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        n2[a] = fma(U[2][a], U[2][a], fma(U[1][a], U[1][a], U[0][a] * U[0][a]));
        R[a] = n2[a] > 0.0 ? rsqrt_acc(n2[a]) : 0.0;
        S[a] = n2[a] * R[a];
#pragma unroll
        for (int r = 0; r < 3; ++r) U[r][a] *= R[a];
    }
    const double lo = fmin(n2[0], fmin(n2[1], n2[2])), hi = fmax(n2[0], fmax(n2[1], n2[2]));
    if (det < 0.0) {
        const int m = n2[0] == lo ? 0 : (n2[1] == lo ? 1 : 2);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (a == m) {
                S[a] = -S[a];
                R[a] = -R[a];
            }
    }
    return lo > 1e-10 * hi;
}

// a unit vector across u
__device__ __forceinline__ void across(const double (&u)[3], double (&v)[3]) {
    const bool x = fabs(u[0]) < 0.6;
    const double d = x ? u[0] : u[1];
    double n = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        v[i] = (i == (x ? 0 : 1) ? 1.0 : 0.0) - d * u[i];
        n = fma(v[i], v[i], n);
    }
    n = rsqrt_acc(n);
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] *= n;
}

__device__ __forceinline__ double pick(const double (&x)[3], int i) { return i == 0 ? x[0] : (i == 1 ? x[1] : x[2]); }

// where principal_axes returned false: the smallest singular value's directions,
// u and v alike, completed to right-handed bases from the other two; of those the
// smaller one's v orthogonal to the larger one's, or, where it too is rounding
// noise of the larger (a lower rank: u not across the larger one's, or F^T u not
// S long and across), any vectors across.  R as principal_axes left it (0 for S =
// 0); i is the smallest, (i, j, k) cyclic.
__device__ __forceinline__ void principal_axes_singular(const float (&F)[3][3], const double (&R)[3],
                                                        double (&U)[3][3], double (&V)[3][3]) {
    double S[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) S[a] = R[a] != 0.0 ? 1.0 / fabs(R[a]) : 0.0;
    const int i = S[0] <= S[1] && S[0] <= S[2] ? 0 : (S[1] <= S[2] ? 1 : 2), j = i == 2 ? 0 : i + 1,
              k = j == 2 ? 0 : j + 1;
    const bool kl = pick(S, k) >= pick(S, j);   // k is the larger of the two
    const double sl = pick(S, kl ? k : j), ss = pick(S, kl ? j : k);
    double ul[3], us[3], vl[3], vs[3];
    double nl = 0.0, ns = 0.0, d = 0.0, e = 0.0;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        ul[r] = pick(U[r], kl ? k : j);
        us[r] = pick(U[r], kl ? j : k);
    }
    if (!(sl > 0.0)) {   // F = 0
        ul[0] = 1.0;
        ul[1] = ul[2] = 0.0;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        vl[c] = sl > 0.0 ? F[0][c] * ul[0] + F[1][c] * ul[1] + F[2][c] * ul[2] : ul[c];
        vs[c] = F[0][c] * us[0] + F[1][c] * us[1] + F[2][c] * us[2];
        nl += vl[c] * vl[c];
    }
    nl = rsqrt_acc(nl);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        vl[c] *= nl;
        d += vs[c] * vl[c];
        e += us[c] * ul[c];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        vs[c] -= d * vl[c];
        ns += vs[c] * vs[c];
    }
    if (fabs(e) < 1e-10 && fabs(d) <= 1e4 * ss && ns > 0.25 * (ss * ss)) {
        ns = rsqrt_acc(ns);
#pragma unroll
        for (int c = 0; c < 3; ++c) vs[c] *= ns;
    } else {
        across(ul, us);
        across(vl, vs);
    }
    double uj[3], uk[3], vj[3], vk[3], ui[3], vi[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        uj[r] = kl ? us[r] : ul[r];
        uk[r] = kl ? ul[r] : us[r];
        vj[r] = kl ? vs[r] : vl[r];
        vk[r] = kl ? vl[r] : vs[r];
    }
    ui[0] = uj[1] * uk[2] - uj[2] * uk[1];
    ui[1] = uj[2] * uk[0] - uj[0] * uk[2];
    ui[2] = uj[0] * uk[1] - uj[1] * uk[0];
    vi[0] = vj[1] * vk[2] - vj[2] * vk[1];
    vi[1] = vj[2] * vk[0] - vj[0] * vk[2];
    vi[2] = vj[0] * vk[1] - vj[1] * vk[0];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            U[r][a] = a == i ? ui[r] : (a == j ? uj[r] : uk[r]);
            V[r][a] = a == i ? vi[r] : (a == j ? vj[r] : vk[r]);
        }
}

}  // namespace mpmx
