// Line transforms held in registers, shared by the Ewald convolution and the
// correlation sampling.
#pragma once
#include "snh_internal.h"

namespace snh {

template <typename T>
struct C2 {
    T re, im;
};

template <typename T>
__device__ __forceinline__ C2<T> cmul2(C2<T> a, C2<T> b)
{
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// ---------------------------------------------------------------------------
// One line of the 3D transform.  Lengths up to kLmax without a prime factor
// above 13 are transformed in registers by Cooley-Tukey steps unrolled at
// compile time (radix 4, then the smallest prime factor; a prime by the
// symmetric sums of its pairs x_j +- x_(p-j)), with every twiddle factor a
// literal.  The primes 17, 19, 23, 29 and 31 go through a direct DFT over LDS
// with the table tw[m] = exp(sign 2 pi i m / L), m < L.
//
// An in-register line reads and writes each value once; the direct DFT, which
// every length but the powers of two took before, reads LDS 2 L times a value:
// the field of one dipolar pyrochlore replica of 15 x 11 x 13 cells 67.6 -> 23.5
// us, of 20 replicas of 15 x 15 x 16 cells 246 -> 66 us, in FP64 of 4 replicas of
// 10 x 10 x 12 cells 88 -> 38 us; one 16^3 replica is the same.

// cos and sin of 2 pi m / L, m < L.
struct CosSin {
    double c, s;
};

constexpr CosSin unit_root(int m, int L)
{
    const int e = 8 * m / L;        // octant
    const int q = (e + 1) / 2 % 4;  // nearest multiple of pi/2: the series run over |x| <= pi/4
    const double x = 6.283185307179586476925286766559 * (double)(8 * m - 2 * ((e + 1) / 2) * L) / (8.0 * L);
    double c = 1, s = x, tc = 1, ts = x;
    for (int k = 1; k <= 10; k++) {
        tc *= -x * x / ((2 * k - 1) * (2 * k));
        ts *= -x * x / ((2 * k) * (2 * k + 1));
        c += tc;
        s += ts;
    }
    if (q == 0) return {c, s};
    if (q == 1) return {-s, c};
    if (q == 2) return {-c, -s};
    return {s, -c};
}

template <int L>
struct Roots {
    double c[L], s[L];
    constexpr Roots() : c(), s()
    {
        for (int m = 0; m < L; m++) {
            c[m] = unit_root(m, L).c;
            s[m] = unit_root(m, L).s;
        }
    }
};

constexpr int fft_radix(int L)
{
    if (L % 4 == 0) return 4;
    for (int p = 2; p * p <= L; p++)
        if (L % p == 0) return p;
    return L;
}

// x <- sum_m x_m exp(S 2 pi i k m / L), in natural order.
template <typename T, int L, int S>
__device__ __forceinline__ void dft_regs(C2<T> (&x)[L])
{
    if constexpr (L == 1) {
        return;
    } else if constexpr (L == 2) {
        const C2<T> a = x[0], b = x[1];
        x[0] = {a.re + b.re, a.im + b.im};
        x[1] = {a.re - b.re, a.im - b.im};
    } else if constexpr (L == 4) {
        const C2<T> a = {x[0].re + x[2].re, x[0].im + x[2].im}, b = {x[0].re - x[2].re, x[0].im - x[2].im};
        const C2<T> c = {x[1].re + x[3].re, x[1].im + x[3].im}, d = {x[1].re - x[3].re, x[1].im - x[3].im};
        x[0] = {a.re + c.re, a.im + c.im};
        x[2] = {a.re - c.re, a.im - c.im};
        x[1] = {b.re - S * d.im, b.im + S * d.re};  // b + S i d
        x[3] = {b.re + S * d.im, b.im - S * d.re};
    } else if constexpr (fft_radix(L) == L) {  // an odd prime
        constexpr Roots<L> w;
        constexpr int H = L / 2;
        C2<T> p[H], m[H];
        C2<T> sum = x[0];
#pragma unroll
        for (int j = 0; j < H; j++) {
            p[j] = {x[j + 1].re + x[L - 1 - j].re, x[j + 1].im + x[L - 1 - j].im};
            m[j] = {x[j + 1].re - x[L - 1 - j].re, x[j + 1].im - x[L - 1 - j].im};
            sum = {sum.re + p[j].re, sum.im + p[j].im};
        }
        const C2<T> x0 = x[0];
        x[0] = sum;
#pragma unroll
        for (int k = 1; k <= H; k++) {
            C2<T> a = x0, b = {(T)0, (T)0};
#pragma unroll
            for (int j = 0; j < H; j++) {
                const T c = (T)w.c[(j + 1) * k % L], s = (T)(S * w.s[(j + 1) * k % L]);
                a = {a.re + c * p[j].re, a.im + c * p[j].im};
                b = {b.re + s * m[j].re, b.im + s * m[j].im};
            }
            x[k] = {a.re - b.im, a.im + b.re};  // a + i b
            x[L - k] = {a.re + b.im, a.im - b.re};
        }
    } else {
        constexpr int P = fft_radix(L), Q = L / P;
        constexpr Roots<L> w;
        C2<T> y[P][Q];
#pragma unroll
        for (int r = 0; r < P; r++) {
#pragma unroll
            for (int m = 0; m < Q; m++) y[r][m] = x[P * m + r];
            dft_regs<T, Q, S>(y[r]);
        }
#pragma unroll
        for (int k = 0; k < Q; k++) {
            C2<T> t[P];
            t[0] = y[0][k];
#pragma unroll
            for (int r = 1; r < P; r++)
                t[r] = k == 0 ? y[r][0] : cmul2(y[r][k], C2<T>{(T)w.c[r * k], (T)(S * w.s[r * k])});
            dft_regs<T, P, S>(t);
#pragma unroll
            for (int q = 0; q < P; q++) x[k + Q * q] = t[q];
        }
    }
}

// Every length up to kLineShort is transformed in registers; kernels whose
// lines are no longer (kMax) leave the longer codelets out, whose registers
// would cost them occupancy.
constexpr int kLineShort = 16;

// Calls f(LineLength<L>) for a length transformed in registers; false for
// the others.
template <int L>
struct LineLength {
    static constexpr int value = L;
};

template <int kMax, typename F>
__device__ __forceinline__ bool with_line_length(int L, F f)
{
#define SNH_LINE(N)         \
    case N:                 \
        f(LineLength<N>{}); \
        return true;
    switch (L) {
        SNH_LINE(1) SNH_LINE(2) SNH_LINE(3) SNH_LINE(4) SNH_LINE(5) SNH_LINE(6) SNH_LINE(7) SNH_LINE(8)
        SNH_LINE(9) SNH_LINE(10) SNH_LINE(11) SNH_LINE(12) SNH_LINE(13) SNH_LINE(14) SNH_LINE(15) SNH_LINE(16)
    }
    if constexpr (kMax > kLineShort) {
        switch (L) {
            SNH_LINE(18) SNH_LINE(20) SNH_LINE(21) SNH_LINE(22) SNH_LINE(24) SNH_LINE(25) SNH_LINE(26)
            SNH_LINE(27) SNH_LINE(28) SNH_LINE(30) SNH_LINE(32)
        }
    }
#undef SNH_LINE
    return false;
}

// Direct DFT of a line of any length L <= kLmax, in place: inputs are read
// from LDS for every output, outputs held in registers until all are formed.
template <typename T>
__device__ __forceinline__ void line_c2c_any(C2<T>* buf, int base, int stride, int L, const C2<T>* tw)
{
    C2<T> out[kLmax];
#pragma unroll
    for (int k = 0; k < kLmax; k++) {
        if (k < L) {
            T ar = 0, ai = 0;
            int m = 0;
            for (int x = 0; x < L; x++) {
                const C2<T> v = buf[base + x * stride], w = tw[m];
                ar += v.re * w.re - v.im * w.im;
                ai += v.re * w.im + v.im * w.re;
                m += k;
                if (m >= L) m -= L;
            }
            out[k] = {ar, ai};
        }
    }
#pragma unroll
    for (int k = 0; k < kLmax; k++)
        if (k < L) buf[base + k * stride] = out[k];
}

// c2c transforms (sign S) of `n` lines: line l holds the L values
// buf[base(l) + x stride], transformed in place, one thread a line.
template <int kMax, int S, typename T, typename Base>
__device__ __forceinline__ void lines_c2c(C2<T>* buf, int n, Base base, int stride, int L, const C2<T>* tw)
{
    const bool regs = with_line_length<kMax>(L, [&](auto len) __attribute__((always_inline)) {
        constexpr int N = decltype(len)::value;
        if constexpr (N > 1)
            for (int l = threadIdx.x; l < n; l += blockDim.x) {
                C2<T>* b = buf + base(l);
                C2<T> x[N];
#pragma unroll
                for (int i = 0; i < N; i++) x[i] = b[i * stride];
                dft_regs<T, N, S>(x);
#pragma unroll
                for (int i = 0; i < N; i++) b[i * stride] = x[i];
            }
    });
    if (kMax > kLineShort && !regs)
        for (int l = threadIdx.x; l < n; l += blockDim.x) line_c2c_any<T>(buf + base(l), 0, stride, L, tw);
}

// Real lines in(l)[0..L) -> half spectra out(l)[0..L/2] (forward).  A line may
// share its storage with its spectrum: in every form a thread holds all
// outputs of its line until it has read the last input.
template <int kMax, typename T, typename In, typename Out>
__device__ __forceinline__ void lines_r2c(int n, In in, Out out, int L, const C2<T>* tw)
{
    const bool regs = with_line_length<kMax>(L, [&](auto len) __attribute__((always_inline)) {
        constexpr int N = decltype(len)::value;
        for (int l = threadIdx.x; l < n; l += blockDim.x) {
            const T* fin = in(l);
            C2<T> x[N];
#pragma unroll
            for (int i = 0; i < N; i++) x[i] = {fin[i], (T)0};
            dft_regs<T, N, -1>(x);
            C2<T>* o = out(l);
#pragma unroll
            for (int k = 0; k <= N / 2; k++) o[k] = x[k];
        }
    });
    if (kMax <= kLineShort || regs) return;
    for (int l = threadIdx.x; l < n; l += blockDim.x) {
        const T* fin = in(l);
        C2<T> o[kLmax / 2 + 1];
#pragma unroll
        for (int k = 0; k <= kLmax / 2; k++) {
            if (k > L / 2) continue;
            T ar = 0, ai = 0;
            int m = 0;
            for (int x = 0; x < L; x++) {
                const T v = fin[x];
                ar += v * tw[m].re;
                ai += v * tw[m].im;
                m += k;
                if (m >= L) m -= L;
            }
            o[k] = {ar, ai};
        }
        C2<T>* po = out(l);
#pragma unroll
        for (int k = 0; k <= kLmax / 2; k++)
            if (k <= L / 2) po[k] = o[k];
    }
}

// Half spectra in(l)[0..L/2] -> real lines out(l)[0..L) (backward, unscaled):
// the real part of the inverse transform of the Hermitian extension
// X[L-k] = conj(X[k]); imaginary parts of X[0] and X[L/2] drop out, as c2r.
// A line may share its storage with its spectrum, as above.
template <int kMax, typename T, typename In, typename Out>
__device__ __forceinline__ void lines_c2r(int n, In in, Out out, int L, const C2<T>* tw)
{
    const bool regs = with_line_length<kMax>(L, [&](auto len) __attribute__((always_inline)) {
        constexpr int N = decltype(len)::value;
        for (int l = threadIdx.x; l < n; l += blockDim.x) {
            const C2<T>* fin = in(l);
            C2<T> x[N];
#pragma unroll
            for (int k = 0; k <= N / 2; k++) x[k] = fin[k];
            if constexpr (N > 2) {
#pragma unroll
                for (int k = N / 2 + 1; k < N; k++) x[k] = {x[N - k].re, -x[N - k].im};
            }
            dft_regs<T, N, 1>(x);
            T* o = out(l);
#pragma unroll
            for (int i = 0; i < N; i++) o[i] = x[i].re;
        }
    });
    if (kMax <= kLineShort || regs) return;
    for (int l = threadIdx.x; l < n; l += blockDim.x) {
        const C2<T>* fin = in(l);
        T o[kLmax];
#pragma unroll
        for (int x = 0; x < kLmax; x++) {
            if (x >= L) continue;
            T acc = 0;
            int m = 0;  // k x mod L
            for (int k = 0; k < L; k++) {
                const C2<T> X = k <= L / 2 ? fin[k] : C2<T>{fin[L - k].re, -fin[L - k].im};
                acc += X.re * tw[m].re - X.im * tw[m].im;
                m += x;
                if (m >= L) m -= L;
            }
            o[x] = acc;
        }
        T* po = out(l);
#pragma unroll
        for (int x = 0; x < kLmax; x++)
            if (x < L) po[x] = o[x];
    }
}

template <typename T>
__device__ __forceinline__ void make_twiddles(C2<T>* tw, int L, int sign)
{
    for (int m = threadIdx.x; m < L; m += blockDim.x) {
        double s, c;
        sincospi(2.0 * m / L, &s, &c);
        tw[m] = {(T)c, (T)(sign * s)};
    }
}

}  // namespace snh
