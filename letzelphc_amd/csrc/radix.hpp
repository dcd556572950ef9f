// radix.hpp -- register DFTs of small lengths for the two-stage line
// transforms of conv.hpp.
//
// A line of N points is N = R1 x R2 (Cooley-Tukey): R2 transforms of length
// R1 over points R2 apart, the twiddles w_N^(j k1), R1 transforms of length
// R2.  Both factors stay in registers, so a line costs one LDS exchange
// whatever N is.  Lengths 2, 3, 4, 5 and 7 are written out; 6, 10, 12, 15
// and 18 are products of coprime factors (Good-Thomas: index maps only, no
// twiddles); 8, 9 and 16 carry constant twiddles.  SIGN +1 is e^{+i}.
#pragma once

#include "common.hpp"

template <int SIGN, typename T>
__device__ __forceinline__ cpx<T> rx_si(cpx<T> a) // SIGN i a
{
    return SIGN > 0 ? cpx<T>{-a.y, a.x} : cpx<T>{a.y, -a.x};
}

// a (c + SIGN i s)
template <int SIGN, typename T>
__device__ __forceinline__ cpx<T> rx_mul(cpx<T> a, double c, double s)
{
    const T tc = (T)c, ts = (T)(SIGN > 0 ? s : -s);
    return {a.x * tc - a.y * ts, a.x * ts + a.y * tc};
}

template <typename T, int SIGN, int R>
struct Rdft;

template <typename T, int SIGN>
struct Rdft<T, SIGN, 1>
{
    static __device__ __forceinline__ void run(cpx<T>*) {}
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 2>
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        const cpx<T> a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 3>
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        const T s = (T)0.86602540378443864676;
        const cpx<T> t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
        const cpx<T> m = {v[0].x - (T)0.5 * t1.x, v[0].y - (T)0.5 * t1.y};
        const cpx<T> i = rx_si<SIGN, T>(cpx<T>{s * t2.x, s * t2.y});
        v[0] = cadd(v[0], t1);
        v[1] = cadd(m, i);
        v[2] = csub(m, i);
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 4>
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        const cpx<T> a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
        const cpx<T> c = cadd(v[1], v[3]), d = rx_si<SIGN, T>(csub(v[1], v[3]));
        v[0] = cadd(a, c);
        v[2] = csub(a, c);
        v[1] = cadd(b, d);
        v[3] = csub(b, d);
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 5>
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
        const cpx<T> t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
        const cpx<T> t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
        const cpx<T> m1 = {v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y};
        const cpx<T> m2 = {v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y};
        const cpx<T> n1 =
            rx_si<SIGN, T>(cpx<T>{s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y});
        const cpx<T> n2 =
            rx_si<SIGN, T>(cpx<T>{s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y});
        v[0] = cadd(v[0], cadd(t1, t2));
        v[1] = cadd(m1, n1);
        v[4] = csub(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 7>
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        const T c[3] = {(T)0.62348980185873353053, (T)-0.22252093395631440429,
                        (T)-0.90096886790241912624};
        const T s[3] = {(T)0.78183148246802980871, (T)0.97492791218182360702,
                        (T)0.43388373911755812048};
        cpx<T> p[3], m[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
        {
            p[i] = cadd(v[1 + i], v[6 - i]);
            m[i] = csub(v[1 + i], v[6 - i]);
        }
        const cpx<T> v0 = v[0];
        v[0] = cadd(v0, cadd(p[0], cadd(p[1], p[2])));
#pragma unroll
        for (int k = 1; k <= 3; ++k)
        {
            cpx<T> a = v0, b = {0, 0};
#pragma unroll
            for (int i = 1; i <= 3; ++i)
            {
                // cos / sin of 2 pi i k / 7 from the first three multiples
                const int e = (i * k) % 7;
                const T ce = c[(e <= 3 ? e : 7 - e) - 1];
                const T se = e <= 3 ? s[e - 1] : -s[7 - e - 1];
                a.x += ce * p[i - 1].x;
                a.y += ce * p[i - 1].y;
                b.x += se * m[i - 1].x;
                b.y += se * m[i - 1].y;
            }
            b = rx_si<SIGN, T>(b);
            v[k] = cadd(a, b);
            v[7 - k] = csub(a, b);
        }
    }
};

// inverse of a modulo m (coprime, small)
constexpr int rx_inv(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if ((a * x) % m == 1) return x;
    return 1;
}

// A, B coprime: x[(B n1 + A n2) mod N] -> X[(B B' k1 + A A' k2) mod N] with
// B B' = 1 mod A, A A' = 1 mod B
template <typename T, int SIGN, int A, int B>
struct RdftGT
{
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        constexpr int N = A * B, IB = rx_inv(B % A, A), IA = rx_inv(A % B, B);
        cpx<T> w[B][A];
#pragma unroll
        for (int b = 0; b < B; ++b)
        {
#pragma unroll
            for (int a = 0; a < A; ++a) w[b][a] = v[(B * a + A * b) % N];
            Rdft<T, SIGN, A>::run(w[b]);
        }
#pragma unroll
        for (int a = 0; a < A; ++a)
        {
            cpx<T> u[B];
#pragma unroll
            for (int b = 0; b < B; ++b) u[b] = w[b][a];
            Rdft<T, SIGN, B>::run(u);
#pragma unroll
            for (int b = 0; b < B; ++b) v[(B * IB * a + A * IA * b) % N] = u[b];
        }
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 6> : RdftGT<T, SIGN, 2, 3>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 10> : RdftGT<T, SIGN, 2, 5>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 12> : RdftGT<T, SIGN, 4, 3>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 15> : RdftGT<T, SIGN, 3, 5>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 18> : RdftGT<T, SIGN, 2, 9>
{
};

// v e^{SIGN 2 pi i K / N} for the constant twiddles of 8, 9 and 16
template <typename T, int SIGN, int N, int K>
__device__ __forceinline__ cpx<T> rx_tw(cpx<T> a)
{
    if constexpr (K % N == 0)
        return a;
    else if constexpr (N == 9)
    {
        constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5,
                                 -0.93969262078590838405};
        constexpr double s[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937,
                                 0.86602540378443864676, 0.34202014332566873304};
        return rx_mul<SIGN, T>(a, c[K], s[K]);
    }
    else
    {
        // sixteenths of a turn
        constexpr int E = K * (16 / N);
        constexpr double c[10] = {1.0,
                                  0.92387953251128675613,
                                  0.70710678118654752440,
                                  0.38268343236508977173,
                                  0.0,
                                  -0.38268343236508977173,
                                  -0.70710678118654752440,
                                  -0.92387953251128675613,
                                  -1.0,
                                  -0.92387953251128675613};
        constexpr double s[10] = {0.0,
                                  0.38268343236508977173,
                                  0.70710678118654752440,
                                  0.92387953251128675613,
                                  1.0,
                                  0.92387953251128675613,
                                  0.70710678118654752440,
                                  0.38268343236508977173,
                                  0.0,
                                  -0.38268343236508977173};
        if constexpr (E == 4)
            return rx_si<SIGN, T>(a);
        else
            return rx_mul<SIGN, T>(a, c[E], s[E]);
    }
}

// A x B with constant twiddles: x[n1 B + n2] -> X[k1 + A k2]
template <typename T, int SIGN, int A, int B>
struct RdftCT
{
    template <int N2, int K1>
    static __device__ __forceinline__ void twiddle(cpx<T> (&w)[B][A])
    {
        if constexpr (N2 < B)
        {
            w[N2][K1] = rx_tw<T, SIGN, A * B, N2 * K1>(w[N2][K1]);
            if constexpr (K1 + 1 < A)
                twiddle<N2, K1 + 1>(w);
            else
                twiddle<N2 + 1, 1>(w);
        }
    }
    static __device__ __forceinline__ void run(cpx<T>* v)
    {
        cpx<T> w[B][A];
#pragma unroll
        for (int b = 0; b < B; ++b)
        {
#pragma unroll
            for (int a = 0; a < A; ++a) w[b][a] = v[a * B + b];
            Rdft<T, SIGN, A>::run(w[b]);
        }
        twiddle<1, 1>(w);
#pragma unroll
        for (int a = 0; a < A; ++a)
        {
            cpx<T> u[B];
#pragma unroll
            for (int b = 0; b < B; ++b) u[b] = w[b][a];
            Rdft<T, SIGN, B>::run(u);
#pragma unroll
            for (int b = 0; b < B; ++b) v[a + A * b] = u[b];
        }
    }
};

template <typename T, int SIGN>
struct Rdft<T, SIGN, 8> : RdftCT<T, SIGN, 2, 4>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 9> : RdftCT<T, SIGN, 3, 3>
{
};
template <typename T, int SIGN>
struct Rdft<T, SIGN, 16> : RdftCT<T, SIGN, 4, 4>
{
};

// Line lengths with a two-stage form and their factors R1 x R2, R1 <= R2:
// the products of 2, 3, 5 and 7 that plane-wave codes choose, both factors
// at most 18.
#define RX_LENGTHS(X)                                                                             \
    X(12, 3, 4) X(14, 2, 7) X(15, 3, 5) X(16, 4, 4) X(18, 3, 6) X(20, 4, 5) X(21, 3, 7)           \
    X(24, 4, 6) X(25, 5, 5) X(27, 3, 9) X(28, 4, 7) X(30, 5, 6) X(32, 4, 8) X(35, 5, 7)           \
    X(36, 6, 6) X(40, 5, 8) X(42, 6, 7) X(45, 5, 9) X(48, 6, 8) X(50, 5, 10) X(54, 6, 9)          \
    X(56, 7, 8) X(60, 6, 10) X(63, 7, 9) X(64, 8, 8) X(70, 7, 10) X(72, 8, 9) X(75, 5, 15)        \
    X(80, 8, 10) X(81, 9, 9) X(84, 7, 12) X(90, 9, 10) X(96, 8, 12) X(100, 10, 10)                \
    X(105, 7, 15) X(108, 9, 12) X(112, 7, 16) X(120, 10, 12) X(126, 7, 18) X(128, 8, 16)          \
    X(135, 9, 15) X(144, 12, 12) X(150, 10, 15) X(160, 10, 16) X(162, 9, 18) X(180, 12, 15)       \
    X(192, 12, 16) X(216, 12, 18) X(225, 15, 15) X(240, 15, 16)

static inline bool rx_factors(int64_t n, int* r1, int* r2)
{
    switch (n)
    {
#define RX_CASE(N, A, B)                                                                          \
    case N:                                                                                       \
        *r1 = A;                                                                                  \
        *r2 = B;                                                                                  \
        return true;
        RX_LENGTHS(RX_CASE)
#undef RX_CASE
        default: return false;
    }
}

// lengths N of the N x N planes with a kernel of their own (conv.hpp)
#define RX_SQUARES(X)                                                                             \
    X(12, 3, 4) X(15, 3, 5) X(16, 4, 4) X(18, 3, 6) X(20, 4, 5) X(24, 4, 6) X(25, 5, 5)           \
    X(27, 3, 9) X(28, 4, 7) X(30, 5, 6) X(32, 4, 8) X(36, 6, 6) X(40, 5, 8) X(42, 6, 7)           \
    X(45, 5, 9) X(48, 6, 8) X(50, 5, 10) X(54, 6, 9) X(56, 7, 8) X(60, 6, 10) X(64, 8, 8)         \
    X(70, 7, 10) X(72, 8, 9) X(75, 5, 15) X(80, 8, 10) X(81, 9, 9) X(84, 7, 12) X(90, 9, 10)      \
    X(96, 8, 12) X(100, 10, 10) X(108, 9, 12) X(120, 10, 12)

// waves per block of a square plane
template <typename T>
constexpr int rx_square_waves(int n)
{
    return sizeof(T) == 4 ? (n >= 72 ? 12 : 4) : n >= 54 ? 8 : 4;
}

static inline bool rx_square(int64_t ny, int64_t nz)
{
    if (ny != nz) return false;
    switch (ny)
    {
#define RX_CASE(N, A, B) case N:
        RX_SQUARES(RX_CASE)
#undef RX_CASE
        return true;
        default: return false;
    }
}
