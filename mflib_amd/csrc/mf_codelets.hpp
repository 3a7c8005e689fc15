// Register DFT codelets (radix 4, 8, 16) and the Stockham pass index rule.
//
// Host+device code so the codelets can be unit-tested on the CPU.  The
// constants are cos/sin of multiples of pi/8 (the 16th roots of unity).
#pragma once
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define MF_HD __host__ __device__ __forceinline__
#else
#define MF_HD inline
#endif

namespace mfcl {

template <typename T>
struct C2 {
    T x, y;
};

template <typename T>
MF_HD C2<T> add(C2<T> a, C2<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
MF_HD C2<T> sub(C2<T> a, C2<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
MF_HD C2<T> mul(C2<T> a, C2<T> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
template <typename T>
MF_HD C2<T> conj(C2<T> a) { return {a.x, -a.y}; }
// multiply by -i (forward) or +i (inverse)
template <bool INV, typename T>
MF_HD C2<T> rotq(C2<T> a)
{
    if constexpr (INV) { return {-a.y, a.x}; }
    return {a.y, -a.x};
}

constexpr double kCos8 = 0.92387953251128675613;   // cos(pi/8)
constexpr double kTan8 = 0.41421356237309504880;   // tan(pi/8)
constexpr double kHalfRt = 0.70710678118654752440; // cos(pi/4)

// a (1 -+ i t) (sign by INV): a rotation by -+ atan(t) up to the factor
// cos(atan(t)), which the caller folds into its next additions.
template <bool INV, typename T>
MF_HD C2<T> rotT(C2<T> a, T t)
{
    if constexpr (INV) { return {a.x - t * a.y, a.y + t * a.x}; }
    return {a.x + t * a.y, a.y - t * a.x};
}
template <typename T>
MF_HD C2<T> addScaled(C2<T> a, T c, C2<T> b) { return {a.x + c * b.x, a.y + c * b.y}; }

template <bool INV, typename T>
MF_HD void dft4(C2<T> &a0, C2<T> &a1, C2<T> &a2, C2<T> &a3)
{
    const C2<T> t0 = add(a0, a2), t1 = sub(a0, a2);
    const C2<T> t2 = add(a1, a3), t3 = rotq<INV>(sub(a1, a3));
    a0 = add(t0, t2);
    a2 = sub(t0, t2);
    a1 = add(t1, t3);
    a3 = sub(t1, t3);
}

// Second stage of the radix-8 and radix-16 codelets: a 4-point DFT of
// a0, c2 a2 and c a1, c a3 with real factors c, c2 left over by rotT.  The
// factors ride on the additions as fused multiply-adds.
template <bool INV, typename T>
MF_HD void dft4Scaled(C2<T> &a0, C2<T> &a1, C2<T> &a2, C2<T> &a3, T c, T c2)
{
    const C2<T> t0 = addScaled(a0, c2, a2), t1 = addScaled(a0, -c2, a2);
    const C2<T> t2 = add(a1, a3), t3 = rotq<INV>(sub(a1, a3));
    a0 = addScaled(t0, c, t2);
    a2 = addScaled(t0, -c, t2);
    a1 = addScaled(t1, c, t3);
    a3 = addScaled(t1, -c, t3);
}

// 8-point DFT in place (natural order in and out).
template <bool INV, typename T>
MF_HD void dft8(C2<T> *v)
{
    C2<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    C2<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4<INV>(e0, e1, e2, e3);
    dft4<INV>(o0, o1, o2, o3);
    const T h = static_cast<T>(kHalfRt);
    // W8^1 o1 and W8^3 o3 without their factor h, W8^2 o2
    const C2<T> p1 = rotT<INV>(o1, T(1));
    const C2<T> p2 = rotq<INV>(o2);
    const C2<T> p3 = rotq<INV>(rotT<INV>(o3, T(1)));
    v[0] = add(e0, o0);
    v[4] = sub(e0, o0);
    v[1] = addScaled(e1, h, p1);
    v[5] = addScaled(e1, -h, p1);
    v[2] = add(e2, p2);
    v[6] = sub(e2, p2);
    v[3] = addScaled(e3, h, p3);
    v[7] = addScaled(e3, -h, p3);
}

// 16-point DFT in place: 4 x 4 decomposition (n = 4 n1 + n2, k = k1 + 4 k2).
// The inner twiddles W16^e are tangent rotations (e = 1, 3, 9 by pi/8 up to
// quarter turns, e = 2, 6 by pi/4, e = 4 a quarter turn) whose cosines ride
// on the second stage's additions: 144 instructions instead of 164 with
// full complex products.
template <bool INV, typename T>
MF_HD void dft16(C2<T> *v)
{
    C2<T> a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        a[n2][0] = v[n2];
        a[n2][1] = v[4 + n2];
        a[n2][2] = v[8 + n2];
        a[n2][3] = v[12 + n2];
        dft4<INV>(a[n2][0], a[n2][1], a[n2][2], a[n2][3]);
    }
    const T t = static_cast<T>(kTan8), c = static_cast<T>(kCos8), h = static_cast<T>(kHalfRt);
    // k1 = 1: W^1, W^2, W^3 = -i W^-1 (forward)
    a[1][1] = rotT<INV>(a[1][1], t);
    a[2][1] = rotT<INV>(a[2][1], T(1));
    a[3][1] = rotq<INV>(rotT<!INV>(a[3][1], t));
    // k1 = 2: W^2, W^4 = -i, W^6 = -i W^2
    a[1][2] = rotT<INV>(a[1][2], T(1));
    a[2][2] = rotq<INV>(a[2][2]);
    a[3][2] = rotq<INV>(rotT<INV>(a[3][2], T(1)));
    // k1 = 3: W^3, W^6, W^9 = -W^1
    a[1][3] = rotq<INV>(rotT<!INV>(a[1][3], t));
    a[2][3] = rotq<INV>(rotT<INV>(a[2][3], T(1)));
    a[3][3] = rotT<INV>(C2<T>{-a[3][3].x, -a[3][3].y}, t);
    dft4<INV>(a[0][0], a[1][0], a[2][0], a[3][0]);
    dft4Scaled<INV>(a[0][1], a[1][1], a[2][1], a[3][1], c, h);
    dft4Scaled<INV>(a[0][2], a[1][2], a[2][2], a[3][2], h, T(1));
    dft4Scaled<INV>(a[0][3], a[1][3], a[2][3], a[3][3], c, h);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        v[k1] = a[0][k1];
        v[k1 + 4] = a[1][k1];
        v[k1 + 8] = a[2][k1];
        v[k1 + 12] = a[3][k1];
    }
}

template <int R, bool INV, typename T>
MF_HD void dftR(C2<T> *v)
{
    if constexpr (R == 2) {
        const C2<T> a = v[0], b = v[1];
        v[0] = add(a, b);
        v[1] = sub(a, b);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        dft8<INV>(v);
    } else {
        static_assert(R == 16, "radix");
        dft16<INV>(v);
    }
}

// Stockham pass of radix R, stride Ns over M points: butterfly j reads
// in[j + r M/R], multiplies element r by W_{Ns R}^{r (j mod Ns)}, applies
// the R-point DFT and writes out[(j - j mod Ns) R + j mod Ns + r Ns].
MF_HD int stockhamDst(int j, int Ns, int R, int r)
{
    const int k = j & (Ns - 1);
    return (j - k) * R + k + r * Ns;
}

}  // namespace mfcl
