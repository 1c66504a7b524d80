// In-register DFTs of the lengths 1, 2, 3, 4, 5, 6, 8, 9, 10, 12, 15 and 16, the building
// blocks of the convolution product's row and column transforms. A mesh side n = A B with A
// and B among these lengths is transformed in two steps: x[B j2 + s] -> A-point DFTs over j2
// (one per s), the twiddles e^{-2 pi i s k1 / n}, B-point DFTs over s, giving X[k1 + A k2].
#pragma once
#include <hip/hip_runtime.h>

#include "cplx.hpp"

namespace xatu_dev {

constexpr int kFftMaxSide = 128;  // largest mesh side of the two-step transform

// Factor pairs (A, B), A <= B, of the supported mesh sides: of the pairs of lengths with
// product n the one with the largest A.
#define XATU_FFT_PAIRS(X)                                                                                    \
    X(1, 2) X(1, 3) X(1, 5) X(2, 2) X(2, 3) X(2, 4) X(2, 5) X(3, 3) X(3, 4) X(3, 5) X(3, 6) X(3, 9) X(4, 4) \
    X(4, 5) X(4, 6) X(4, 8) X(5, 5) X(5, 6) X(5, 8) X(5, 9) X(5, 10) X(5, 15) X(6, 6) X(6, 8) X(6, 9)       \
    X(6, 10) X(8, 8) X(8, 9) X(8, 10) X(8, 12) X(8, 16) X(9, 9) X(9, 10) X(9, 12) X(10, 10) X(10, 12)

// (A, B) of a mesh side; A = 0: the side is not one of the supported products.
inline void fft_factors(int n, int& A, int& B) {
    A = B = 0;
#define XATU_TRY(a, b)     \
    if (n == (a) * (b)) { \
        A = (a);           \
        B = (b);           \
        return;            \
    }
    XATU_FFT_PAIRS(XATU_TRY)
#undef XATU_TRY
}

// cos(2 pi a / 720) for 0 <= a <= 180, the angles that the composite lengths use.
__host__ __device__ constexpr double cos_quadrant(int a) {
    switch (a) {
        case 0: return 1.0;
        case 180: return 0.0;
        case 12: return 0.99452189536827333692;
        case 20: return 0.98480775301220805937;
        case 24: return 0.97814760073380563793;
        case 36: return 0.95105651629515357212;
        case 40: return 0.93969262078590838405;
        case 45: return 0.92387953251128675613;
        case 48: return 0.9135454576426008955;
        case 60: return 0.86602540378443864676;
        case 72: return 0.8090169943749474241;
        case 80: return 0.7660444431189780352;
        case 84: return 0.74314482547739423501;
        case 90: return 0.7071067811865475244;
        case 96: return 0.66913060635885821383;
        case 100: return 0.64278760968653932632;
        case 108: return 0.58778525229247312917;
        case 120: return 0.5;
        case 132: return 0.40673664307580020775;
        case 135: return 0.38268343236508977173;
        case 140: return 0.34202014332566873304;
        case 144: return 0.3090169943749474241;
        case 156: return 0.2079116908177593371;
        case 160: return 0.17364817766693034885;
        case 168: return 0.1045284632676534714;

    }
    return 0.0;
}
// cos and sin of 2 pi k / RD (RD a divisor of 720); the arguments are constants after unrolling.
__host__ __device__ constexpr double root_cos(int RD, int k) {
    int a = (k * (720 / RD)) % 720;
    if (a > 360) a = 720 - a;
    return a <= 180 ? cos_quadrant(a) : -cos_quadrant(360 - a);
}
__host__ __device__ constexpr double root_sin(int RD, int k) { return root_cos(720, k * (720 / RD) + 540); }

// e^{SG 2 pi i k / RD} x
template <typename R, int RD, int SG>
__device__ inline cx_t<R> cmul_root(cx_t<R> x, int k) {
    k %= RD;
    if (k == 0) return x;
    if (4 * k == RD) return mk(R(-SG) * x.y, R(SG) * x.x);
    if (2 * k == RD) return mk(-x.x, -x.y);
    if (4 * k == 3 * RD) return mk(R(SG) * x.y, R(-SG) * x.x);
    const R c = static_cast<R>(root_cos(RD, k)), s = static_cast<R>(SG * root_sin(RD, k));
    return mk(c * x.x - s * x.y, c * x.y + s * x.x);
}

// In-register DFT of length RD <= 5, sign SG in the exponent.
template <typename R, int RD, int SG>
__device__ inline void small_dft(cx_t<R> (&v)[RD]) {
    using C = cx_t<R>;
    auto isc = [](C z, R f) { return mk(R(-SG) * f * z.y, R(SG) * f * z.x); };  // i SG f z
    if constexpr (RD == 2) {
        const C a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (RD == 3) {
        const R h3 = R(0.86602540378443864676);  // sin(2 pi / 3)
        const C a = cadd(v[1], v[2]), d = csub(v[1], v[2]);
        const C m = mk(v[0].x - R(0.5) * a.x, v[0].y - R(0.5) * a.y);
        const C t = isc(d, h3);
        v[0] = cadd(v[0], a);
        v[1] = cadd(m, t);
        v[2] = csub(m, t);
    } else if constexpr (RD == 4) {
        const C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]), t2 = cadd(v[1], v[3]), t3 = isc(csub(v[1], v[3]), R(1));
        v[0] = cadd(t0, t2);
        v[1] = cadd(t1, t3);
        v[2] = csub(t0, t2);
        v[3] = csub(t1, t3);
    } else if constexpr (RD == 5) {
        // cos and sin of 2 pi / 5 and 4 pi / 5
        const R c1 = R(0.30901699437494742410), s1 = R(0.95105651629515357212);
        const R c2 = R(-0.80901699437494742410), s2 = R(0.58778525229247312917);
        const C a1 = cadd(v[1], v[4]), d1 = csub(v[1], v[4]), a2 = cadd(v[2], v[3]), d2 = csub(v[2], v[3]);
        const C p1 = mk(v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y);
        const C p2 = mk(v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y);
        const C q1 = isc(mk(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y), R(1));
        const C q2 = isc(mk(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y), R(1));
        v[0] = cadd(v[0], cadd(a1, a2));
        v[1] = cadd(p1, q1);
        v[4] = csub(p1, q1);
        v[2] = cadd(p2, q2);
        v[3] = csub(p2, q2);
    } else {
        static_assert(RD == 1, "radix");
    }
}

// DFT of length A B in registers as two Stockham stages (radix A, then radix B).
template <typename R, int A, int B, int SG>
__device__ inline void composite_dft(cx_t<R> (&v)[A * B]) {
    using C = cx_t<R>;
    constexpr int RD = A * B;
    C t[RD];
#pragma unroll
    for (int j = 0; j < B; ++j) {
        C x[A];
#pragma unroll
        for (int r = 0; r < A; ++r) x[r] = v[j + r * B];
        small_dft<R, A, SG>(x);
#pragma unroll
        for (int r = 0; r < A; ++r) t[j * A + r] = x[r];
    }
#pragma unroll
    for (int j = 0; j < A; ++j) {
        C x[B];
#pragma unroll
        for (int r = 0; r < B; ++r) x[r] = cmul_root<R, RD, SG>(t[j + r * A], j * r);
        small_dft<R, B, SG>(x);
#pragma unroll
        for (int r = 0; r < B; ++r) v[j + r * A] = x[r];
    }
}

// DFT of one of the lengths, sign SG.
template <typename R, int RD, int SG>
__device__ inline void dft_len(cx_t<R> (&a)[RD]) {
    if constexpr (RD <= 5) {
        small_dft<R, RD, SG>(a);
    } else if constexpr (RD == 6) {
        composite_dft<R, 3, 2, SG>(a);
    } else if constexpr (RD == 8) {
        composite_dft<R, 4, 2, SG>(a);
    } else if constexpr (RD == 9) {
        composite_dft<R, 3, 3, SG>(a);
    } else if constexpr (RD == 10) {
        composite_dft<R, 5, 2, SG>(a);
    } else if constexpr (RD == 12) {
        composite_dft<R, 3, 4, SG>(a);
    } else if constexpr (RD == 15) {
        composite_dft<R, 5, 3, SG>(a);
    } else {
        static_assert(RD == 16, "length");
        composite_dft<R, 4, 4, SG>(a);
    }
}

}  // namespace xatu_dev
