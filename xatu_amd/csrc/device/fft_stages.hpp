// In-register DFTs of the lengths 1 to 17, 19, 23, 29 and 31, the building blocks of the
// convolution product's row and column transforms. A mesh side n = A B with A and B among these
// lengths, or 37 and 41 themselves, is transformed in two steps: x[B j2 + s] -> A-point DFTs over j2
// (one per s), the twiddles e^{-2 pi i s k1 / n}, B-point DFTs over s, giving X[k1 + A k2]
// (a prime B much longer than A spread over lanes, conv_rows.hpp). That covers 100 of the 128 sides up to
// 128, all but 125 and those with a longer prime factor; pairs of factors 2, 3 and 5 alone cover 36, and
// the others took the library's transforms over whole meshes (products of 16 vectors, 12 orbitals, with
// their copies from and to the host: FP64 23 x 23 0.45 -> 0.30 ms, 49 x 49 0.96 -> 0.69, 77 x 77 1.72 -> 1.36,
// 119 x 119 4.9 -> 3.8). Longer primes spread over lanes spilled in the column kernel (53 x 53: 1.35 -> 2.9 ms).
#pragma once
#include <hip/hip_runtime.h>

#include "cplx.hpp"

namespace xatu_dev {

constexpr int kFftMaxSide = 128;  // largest mesh side of the two-step transform

// Factor pairs (A, B), A <= B, of the supported mesh sides.
#define XATU_FFT_PAIRS(X)                                                                                     \
    X(1, 1) X(1, 2) X(1, 3) X(1, 5) X(1, 7) X(1, 11) X(1, 13) X(1, 17) X(1, 19) X(1, 23) X(1, 29) X(1, 31)    \
    X(1, 37) X(1, 41) X(2, 2) X(2, 3) X(2, 4) X(2, 5) X(2, 7) X(2, 11) X(2, 13) X(2, 17) X(2, 19) X(2, 23)    \
    X(2, 29) X(2, 31) X(3, 3) X(3, 4) X(3, 5) X(3, 6) X(3, 7) X(3, 9) X(3, 11) X(3, 13) X(3, 17) X(3, 19)     \
    X(3, 23) X(3, 29) X(3, 31) X(4, 4) X(4, 5) X(4, 6) X(4, 7) X(4, 8) X(4, 11) X(4, 13) X(4, 17) X(4, 19)    \
    X(4, 23) X(4, 29) X(4, 31) X(5, 5) X(5, 6) X(5, 7) X(5, 8) X(5, 9) X(5, 10) X(5, 11) X(5, 13) X(5, 15)    \
    X(5, 17) X(5, 19) X(5, 23) X(6, 6) X(6, 7) X(6, 8) X(6, 9) X(6, 10) X(6, 11) X(6, 13) X(6, 17) X(6, 19)   \
    X(7, 7) X(7, 8) X(7, 9) X(7, 10) X(7, 11) X(7, 12) X(7, 13) X(7, 14) X(7, 15) X(7, 17) X(8, 8) X(8, 9)    \
    X(8, 10) X(8, 11) X(8, 12) X(8, 13) X(8, 14) X(8, 16) X(9, 9) X(9, 10) X(9, 11) X(9, 12) X(9, 13)         \
    X(9, 14) X(10, 10) X(10, 11) X(10, 12) X(11, 11)

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
// cos and sin of 2 pi k / p, k = 1 .. (p - 1) / 2
template <int P>
struct PrimeRoots;
template <>
struct PrimeRoots<7> {
    static constexpr double c[3] = {
        0.623489801858733530525, -0.222520933956314404289, -0.900968867902419126236};
    static constexpr double s[3] = {
        0.781831482468029808708, 0.974927912181823607018, 0.433883739117558120476};
};
template <>
struct PrimeRoots<11> {
    static constexpr double c[5] = {
        0.841253532831181168862, 0.415415013001886425529, -0.142314838273285140444, -0.654860733945285064057,
        -0.959492973614497389890};
    static constexpr double s[5] = {
        0.540640817455597582108, 0.909631995354518371412, 0.989821441880932732376, 0.755749574354258283774,
        0.281732556841429697711};
};
template <>
struct PrimeRoots<13> {
    static constexpr double c[6] = {
        0.885456025653209895900, 0.568064746731155802512, 0.120536680255323053349, -0.354604887042535625970,
        -0.748510748171101098635, -0.970941817426052027157};
    static constexpr double s[6] = {
        0.464723172043768545656, 0.822983865893656394580, 0.992708874098053992801, 0.935016242685414823440,
        0.663122658240795202377, 0.239315664287557767149};
};
template <>
struct PrimeRoots<17> {
    static constexpr double c[8] = {
        0.932472229404355804573, 0.739008917220659115925, 0.445738355776538267396, 0.092268359463301995240,
        -0.273662990072082863539, -0.602634636379256389179, -0.850217135729614152134, -0.982973099683901778282};
    static constexpr double s[8] = {
        0.361241666187152948745, 0.673695643646557211713, 0.895163291355062322067, 0.995734176295034521871,
        0.961825643172819070409, 0.798017227280239503333, 0.526432162877355800245, 0.183749517816570331574};
};
template <>
struct PrimeRoots<19> {
    static constexpr double c[9] = {
        0.945817241700634679020, 0.789140509396393599219, 0.546948158122426874712, 0.245485487140799148922,
        -0.082579345472332324600, -0.401695424652969457517, -0.677281571625741074762, -0.879473751206489071391,
        -0.986361303402722373603};
    static constexpr double s[9] = {
        0.324699469204683487408, 0.614212712689667817444, 0.837166478262528574806, 0.969400265939330416736,
        0.996584493006669849819, 0.915773326655057439919, 0.735723910673131624774, 0.475947393037073544431,
        0.164594590280733894144};
};
template <>
struct PrimeRoots<23> {
    static constexpr double c[11] = {
        0.962917287347799295015, 0.854419404546488552548, 0.682553143218654082875, 0.460065037731152126042,
        0.203456013052633789878, -0.068242413364670975921, -0.334879612170986151958, -0.576680322114867141251,
        -0.775711290704419807041, -0.917211301505453017844, -0.990685946036330752342};
    static constexpr double s[11] = {
        0.269796771157024271245, 0.519583950035433578133, 0.730835964278124101651, 0.887885218402375234984,
        0.979084087682322875633, 0.997668769190539198454, 0.942260922118820495618, 0.816969893010442016973,
        0.631087944326052789367, 0.398401089846241457998, 0.136166649096246590761};
};
template <>
struct PrimeRoots<29> {
    static constexpr double c[14] = {
        0.976620555710086683208, 0.907575419670957053620, 0.796093065705643745998, 0.647386284781827639182,
        0.468408440699790139216, 0.267528338529220821195, 0.054138908585417526150, -0.161781996552764726544,
        -0.370138155339914356864, -0.561187065362382369270, -0.725995491923130858138, -0.856857176167589244523,
        -0.947653171182802444274, -0.994137957154359608955};
    static constexpr double s[14] = {
        0.214970440211024067182, 0.419889101560264576974, 0.605174215193765165924, 0.762162055127636463256,
        0.883512044446022922827, 0.963549992519222960043, 0.998533413851123864572, 0.986826522541526151769,
        0.928976719816791441790, 0.827688998156890556136, 0.687699458853423293084, 0.515553857177021739710,
        0.319301530135979973197, 0.108119018423941763031};
};
template <>
struct PrimeRoots<31> {
    static constexpr double c[15] = {
        0.979529941252494493938, 0.918957811620230629127, 0.820763441207276326364, 0.688966919075686567801,
        0.528964010326962457365, 0.347305252844820285542, 0.151427777504576663657, -0.050649168838712712279,
        -0.250652532258720539315, -0.440394151557634309516, -0.612105982547662844147, -0.758758122692790901913,
        -0.874346616144582118827, -0.954139256400048851476, -0.994869323391895146321};
    static constexpr double s[15] = {
        0.201298520088660079142, 0.394355855113318580102, 0.571268215094792279157, 0.724792787229119958865,
        0.848644257494750950464, 0.937752132147080458429, 0.988468324328111399162, 0.998716507171052807146,
        0.968077118866204305153, 0.897804539570741657137, 0.790775736937698582078, 0.651372482722222207454,
        0.485301962531081025215, 0.299363122973357954008, 0.101168321987432177786};
};

// cos and sin of 2 pi k / RD (RD a divisor of 720, or 14); the arguments are constants after unrolling.
__host__ __device__ constexpr double seventh(int k, bool sine) {
    k %= 7;
    if (k == 0) return sine ? 0.0 : 1.0;
    const int m = k <= 3 ? k : 7 - k;
    return sine ? (k <= 3 ? PrimeRoots<7>::s[m - 1] : -PrimeRoots<7>::s[m - 1]) : PrimeRoots<7>::c[m - 1];
}
// a fourteenth root of unity is a seventh one or the negative of one
__host__ __device__ constexpr double fourteenth(int k, bool sine) {
    return k % 2 == 0 ? seventh(k / 2, sine) : -seventh((k + 7) / 2, sine);
}
__host__ __device__ constexpr double root_cos(int RD, int k) {
    if (RD == 14) return fourteenth(k, false);
    int a = (k * (720 / RD)) % 720;
    if (a > 360) a = 720 - a;
    return a <= 180 ? cos_quadrant(a) : -cos_quadrant(360 - a);
}
__host__ __device__ constexpr double root_sin(int RD, int k) {
    return RD == 14 ? fourteenth(k, true) : root_cos(720, k * (720 / RD) + 540);
}

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

// DFT of an odd prime length: the sums and differences of the entries j and P - j meet the cosines
// and the sines, so that it takes (P - 1)^2 real multiply-adds of complex numbers instead of twice as
// many complex ones.
template <typename R, int P, int SG>
__device__ inline void prime_dft(cx_t<R> (&v)[P]) {
    using C = cx_t<R>;
    constexpr int H = (P - 1) / 2;
    C a[H], d[H];
    const C x0 = v[0];
    C sum = x0;
#pragma unroll
    for (int j = 0; j < H; ++j) {
        a[j] = cadd(v[j + 1], v[P - 1 - j]);
        d[j] = csub(v[j + 1], v[P - 1 - j]);
        sum = cadd(sum, a[j]);
    }
    v[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        C p = x0, q = mk(R(0), R(0));
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const int r = j * k % P, m = r <= H ? r : P - r;
            const R c = static_cast<R>(PrimeRoots<P>::c[m - 1]);
            const R s = static_cast<R>(r <= H ? PrimeRoots<P>::s[m - 1] : -PrimeRoots<P>::s[m - 1]);
            p = mk(p.x + c * a[j - 1].x, p.y + c * a[j - 1].y);
            q = mk(q.x + s * d[j - 1].x, q.y + s * d[j - 1].y);
        }
        const C t = mk(R(-SG) * q.y, R(SG) * q.x);
        v[k] = cadd(p, t);
        v[P - k] = csub(p, t);
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
        if constexpr (A == 7) prime_dft<R, A, SG>(x);
        else small_dft<R, A, SG>(x);
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
    } else if constexpr (RD == 7 || RD == 11 || RD == 13 || RD == 17 || RD == 19 || RD == 23 || RD == 29 || RD == 31) {
        prime_dft<R, RD, SG>(a);
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
    } else if constexpr (RD == 14) {
        composite_dft<R, 7, 2, SG>(a);
    } else if constexpr (RD == 15) {
        composite_dft<R, 5, 3, SG>(a);
    } else {
        static_assert(RD == 16, "length");
        composite_dft<R, 4, 4, SG>(a);
    }
}

}  // namespace xatu_dev
