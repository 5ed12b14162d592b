// Complex FFTs of length 64 P run by one wave (FP64): P points per lane in
// registers, three passes (8, 8, P) with two exchanges through the wave's own
// LDS buffer and no block barrier.
//
// With k = k1 + P k2 on the spectral side (k1 < P, k2 = r + 8 s < 64) and n =
// j + 64 q on the grid side (lane j, q < P):
//   inverse  pass A, task (k1, r): 8 points over s, times exp(2 pi i r a / 64)
//            pass B, task (k1, a): 8 points over r, j = a + 8 b
//            pass C, lane j: times exp(2 pi i j k1 / N), P points over k1
//   forward  the same backwards with conjugated factors
// so that after the inverse and before the forward transform lane j holds the
// grid points j + 64 q whatever P is: products of several transformed fields
// are formed in the registers of the lane that owns the point.  The 8 P tasks
// of passes A and B are dealt over the lanes (task = lane + 64 round).
//
// The buffer holds element (k1, i) of the exchanges at 72 k1 + i; the first
// exchange rotates the eight values of a task's row, so that the stores by r
// and the loads by a both touch distinct banks.
#pragma once

#include "mhx_fftcore.h"

namespace mhx {

namespace {

// 8-point DFT as 2 x 4
template <typename C> struct Dft<8, C> {
    __device__ __forceinline__ static void run(C *x, int sign)
    {
        typedef decltype(C::x) T;
        const T h = T(0.70710678118654752440), sg = T(sign);
        C e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
        Dft<4, C>::run(e, sign);
        Dft<4, C>::run(o, sign);
        o[1] = mk<C>(h * (o[1].x - sg * o[1].y), h * (o[1].y + sg * o[1].x));
        o[2] = cmuli(o[2], sign);
        o[3] = mk<C>(-h * (o[3].x + sg * o[3].y), h * (sg * o[3].x - o[3].y));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = cadd(e[k], o[k]);
            x[k + 4] = csub(e[k], o[k]);
        }
    }
};

// 9-point DFT as 3 x 3, n = 3 n1 + n2, k = k1 + 3 k2
template <typename C> struct Dft<9, C> {
    __device__ __forceinline__ static void run(C *x, int sign)
    {
        typedef decltype(C::x) T;
        const T sg = T(sign);
        const T c1 = T(0.76604444311897803520), s1 = sg * T(0.64278760968653932632);
        const T c2 = T(0.17364817766693034885), s2 = sg * T(0.98480775301220805937);
        const T c4 = T(-0.93969262078590838405), s4 = sg * T(0.34202014332566873304);
        C a[3][3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) {
            C t[3] = {x[n2], x[3 + n2], x[6 + n2]};
            Dft<3, C>::run(t, sign);
#pragma unroll
            for (int k1 = 0; k1 < 3; ++k1) a[n2][k1] = t[k1];
        }
        a[1][1] = cmul(a[1][1], mk<C>(c1, s1));
        a[1][2] = cmul(a[1][2], mk<C>(c2, s2));
        a[2][1] = cmul(a[2][1], mk<C>(c2, s2));
        a[2][2] = cmul(a[2][2], mk<C>(c4, s4));
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            C t[3] = {a[0][k1], a[1][k1], a[2][k1]};
            Dft<3, C>::run(t, sign);
#pragma unroll
            for (int k2 = 0; k2 < 3; ++k2) x[k1 + 3 * k2] = t[k2];
        }
    }
};

constexpr int inv_mod(int b, int a)  // b^-1 mod a
{
    for (int i = 1; i < a; ++i)
        if (b * i % a == 1) return i;
    return 1;
}

// A B points, A and B coprime, by the prime-factor index maps (no twiddles)
template <int A, int B, typename C> struct DftPf {
    __device__ __forceinline__ static void run(C *x, int sign)
    {
        constexpr int R = A * B, ka = B * inv_mod(B % A, A) % R, kb = A * inv_mod(A % B, B) % R;
        C y[A][B], out[R];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
            C t[A];
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) t[n1] = x[(B * n1 + A * n2) % R];
            Dft<A, C>::run(t, sign);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) y[k1][n2] = t[k1];
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            Dft<B, C>::run(y[k1], sign);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) out[(ka * k1 + kb * k2) % R] = y[k1][k2];
        }
#pragma unroll
        for (int i = 0; i < R; ++i) x[i] = out[i];
    }
};
template <typename C> struct Dft<1, C> {
    __device__ __forceinline__ static void run(C *, int) {}
};
template <typename C> struct Dft<6, C> : DftPf<2, 3, C> {};
template <typename C> struct Dft<10, C> : DftPf<2, 5, C> {};
template <typename C> struct Dft<15, C> : DftPf<3, 5, C> {};
template <typename C> struct Dft<18, C> : DftPf<2, 9, C> {};
template <typename C> struct Dft<20, C> : DftPf<4, 5, C> {};
template <typename C> struct Dft<24, C> : DftPf<3, 8, C> {};

template <int P> struct WaveFFT {
    typedef double2 C;
    static constexpr int N = 64 * P, TASKS = 8 * P, RND = (TASKS + 63) / 64;
    static constexpr int BUF = 72 * P;  // complex elements of the wave's buffer

    // factors: w64(a) = exp(2 pi i a (lane % 8) / 64), wn(k1) = exp(2 pi i lane k1 / N)
    // x[q] = sum_k Y_k exp(2 pi i k n / N), n = lane + 64 q; y(rd, s, k) gives
    // Y_k, k = k1 + P (lane % 8 + 8 s) of the task of round rd
    template <class W64, class Wn, class Y>
    __device__ __forceinline__ static void inverse(C *buf, int lane, W64 &&w64, Wn &&wn, Y &&y, C *x)
    {
        const int r = lane & 7;
#pragma unroll
        for (int rd = 0; rd < RND; ++rd) {
            const int k1 = (lane + 64 * rd) >> 3;
            if (8 * P % 64 == 0 || rd + 1 < RND || k1 < P) {
                C v[8];
#pragma unroll
                for (int s = 0; s < 8; ++s) v[s] = y(rd, s, k1 + P * (r + 8 * s));
                Dft<8, C>::run(v, +1);
#pragma unroll
                for (int a = 0; a < 8; ++a)
                    buf[72 * k1 + 8 * a + ((r + a) & 7)] = a ? cmul(v[a], w64(a)) : v[a];
            }
        }
        wave_order();
#pragma unroll
        for (int rd = 0; rd < RND; ++rd) {
            const int k1 = (lane + 64 * rd) >> 3, a = r;
            if (8 * P % 64 == 0 || rd + 1 < RND || k1 < P) {
                C v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = buf[72 * k1 + 8 * a + ((i + a) & 7)];
                wave_order();
                Dft<8, C>::run(v, +1);
#pragma unroll
                for (int b = 0; b < 8; ++b) buf[72 * k1 + a + 8 * b] = v[b];
            }
        }
        wave_order();
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) {
            x[k1] = buf[72 * k1 + lane];
            if (k1) x[k1] = cmul(x[k1], wn(k1));
        }
        wave_order();
        Dft<P, C>::run(x, +1);
    }

    // Y_k = sum_n x_n exp(-2 pi i k n / N) from x[q] = x_{lane + 64 q}, left in
    // buf at index k (N elements)
    template <class W64, class Wn>
    __device__ __forceinline__ static void forward(C *buf, int lane, W64 &&w64, Wn &&wn, C *x)
    {
        const int r = lane & 7;
        Dft<P, C>::run(x, -1);
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) buf[72 * k1 + lane] = k1 ? cmul(x[k1], cconj(wn(k1))) : x[k1];
        wave_order();
#pragma unroll
        for (int rd = 0; rd < RND; ++rd) {
            const int k1 = (lane + 64 * rd) >> 3, a = r;
            if (8 * P % 64 == 0 || rd + 1 < RND || k1 < P) {
                C v[8];
#pragma unroll
                for (int b = 0; b < 8; ++b) v[b] = buf[72 * k1 + a + 8 * b];
                wave_order();
                Dft<8, C>::run(v, -1);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    buf[72 * k1 + 8 * a + ((i + a) & 7)] = i ? cmul(v[i], cconj(w64(i))) : v[i];
            }
        }
        wave_order();
        C v[RND][8];
#pragma unroll
        for (int rd = 0; rd < RND; ++rd) {
            const int k1 = (lane + 64 * rd) >> 3;
            if (8 * P % 64 == 0 || rd + 1 < RND || k1 < P) {
#pragma unroll
                for (int a = 0; a < 8; ++a) v[rd][a] = buf[72 * k1 + 8 * a + ((r + a) & 7)];
                Dft<8, C>::run(v[rd], -1);
            }
        }
        wave_order();
#pragma unroll
        for (int rd = 0; rd < RND; ++rd) {
            const int k1 = (lane + 64 * rd) >> 3;
            if (8 * P % 64 == 0 || rd + 1 < RND || k1 < P) {
#pragma unroll
                for (int s = 0; s < 8; ++s) buf[k1 + P * (r + 8 * s)] = v[rd][s];
            }
        }
        wave_order();
    }
};

}  // namespace

}  // namespace mhx
