// Device building blocks for the matched-filter kernels (gfx950 / CDNA4).
//
// FFTs are Stockham auto-sort transforms executed in LDS: each pass reads
// a thread's butterflies into registers, synchronises, applies twiddles and
// a radix-4 (or a final radix-2) DFT and writes back in place.
//
// The correlation of a block of N = 2M real samples is taken modulo
// z^N + 1 (its outputs before the wrap-around are the linear correlation's,
// as with z^N - 1).  z^N + 1 = (z^M + i)(z^M - i), and the second factor's
// residue is the conjugate of the first's, so a real block x is carried by
// the M complex values
//     u_j = (x_j - i x_{j+M}) W_{4M}^j,   W_{4M} = exp(-2 pi i / 4M),
// whose M-point transform U_k holds x at the roots exp(-2 pi i (k+1/4)/M) of
// z^M = -i.  The spectrum of the correlation with a template is U_k H_k, H_k
// the conjugate of the template's own transform over M, with no pairing of
// bins, and its inverse transform times W_{4M}^-n is c_n - i c_{n+M}.  The
// packing of even and odd samples that a transform of z^N - 1 needs (split
// and merge of bins k and M - k around every product) has no counterpart.
//
// Twiddles W_{4M}^e come from a two-level table (64 low entries x 4M/64 high
// entries, computed in FP64 on the host with the C library's cos/sin and
// rounded to T), so one complex product gives any twiddle to about one ulp.
#pragma once
#include <hip/hip_runtime.h>

#include "mf_codelets.hpp"

namespace mfdev {

template <typename T>
using Cx = mfcl::C2<T>;

// Pointers read from descriptor tables are generic; accessing global
// memory through them would compile to FLAT instructions, which also count
// against the LDS wait counter.  These casts make them global.
template <typename T>
using gptr = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ gptr<T> to_global(T *p)
{
    return (gptr<T>)p;
}
template <typename T>
__device__ __forceinline__ gptr<const T> to_global(const T *p)
{
    return (gptr<const T>)p;
}
// Complex element i of a global array (component loads merge into one
// 2-wide access).
template <typename T>
__device__ __forceinline__ Cx<T> load_cx(gptr<const Cx<T>> p, int i)
{
    const gptr<const T> s = (gptr<const T>)p;
    return Cx<T>{s[2 * i], s[2 * i + 1]};
}

// Raw buffer resource over `bytes` bytes from p (stride 0; dword 3 selects
// 32-bit data, as for every gfx9 raw buffer access).  Stores through it at
// byte offsets >= bytes are dropped by the hardware range check, so a
// store needs no branch of its own and every path issues the same
// instructions.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(void *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00020000);
}
__device__ __forceinline__ void buffer_store(float x, __amdgpu_buffer_rsrc_t r, int byteOff)
{
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), r, byteOff, 0, 0);
}
__device__ __forceinline__ void buffer_store(double x, __amdgpu_buffer_rsrc_t r, int byteOff)
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const unsigned long long a = static_cast<unsigned long long>(__double_as_longlong(x));
    const u2 d = {static_cast<unsigned>(a), static_cast<unsigned>(a >> 32)};
    __builtin_amdgcn_raw_buffer_store_b64(d, r, byteOff, 0, 0);
}

template <typename T>
__device__ __forceinline__ Cx<T> cadd(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> csub(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ Cx<T> cconj(Cx<T> a) { return {a.x, -a.y}; }
// i * a
template <typename T>
__device__ __forceinline__ Cx<T> cmuli(Cx<T> a) { return {-a.y, a.x}; }
// -i * a
template <typename T>
__device__ __forceinline__ Cx<T> cmulmi(Cx<T> a) { return {a.y, -a.x}; }

// Two-level twiddle table resident in LDS.
template <typename T>
struct Twiddle {
    const Cx<T> *lo;  // W_{4M}^i,       i < 64
    const Cx<T> *hi;  // W_{4M}^(64 j),  j < 4M/64
    __device__ __forceinline__ Cx<T> operator()(int e) const { return cmul(lo[e & 63], hi[e >> 6]); }
};

template <int R, bool INV, typename T>
__device__ __forceinline__ void dft(Cx<T> *v)
{
    if constexpr (R == 2) {
        Cx<T> a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else {
        static_assert(R == 4, "radix");
        Cx<T> t0 = cadd(v[0], v[2]);
        Cx<T> t1 = csub(v[0], v[2]);
        Cx<T> t2 = cadd(v[1], v[3]);
        Cx<T> d = csub(v[1], v[3]);
        Cx<T> t3 = INV ? cmuli(d) : cmulmi(d);
        v[0] = cadd(t0, t2);
        v[1] = cadd(t1, t3);
        v[2] = csub(t0, t2);
        v[3] = csub(t1, t3);
    }
}

// One Stockham pass of radix R over M points with input stride Ns.
// Every thread of the block must call it (it synchronises twice).
template <typename T, int M, int R, int NT, bool INV>
__device__ __forceinline__ void stockham_pass(Cx<T> *buf, int Ns, Twiddle<T> tw)
{
    constexpr int NB = M / R;
    constexpr int BPT = (NB + NT - 1) / NT;
    const int t = threadIdx.x;
    Cx<T> v[BPT][R];
#pragma unroll
    for (int b = 0; b < BPT; ++b) {
        const int j = t + b * NT;
        if (NB % NT == 0 || j < NB) {
#pragma unroll
            for (int r = 0; r < R; ++r) { v[b][r] = buf[j + r * NB]; }
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < BPT; ++b) {
        const int j = t + b * NT;
        if (NB % NT == 0 || j < NB) {
            const int k = j & (Ns - 1);
            // W_{Ns R}^{r k} = W_{4M}^{r * 4k M / (Ns R)}
            const int step = 4 * (M / (Ns * R)) * k;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                Cx<T> w = tw(r * step);
                if (INV) { w.y = -w.y; }
                v[b][r] = cmul(v[b][r], w);
            }
            dft<R, INV>(v[b]);
            const int idxD = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) { buf[idxD + r * Ns] = v[b][r]; }
        }
    }
    __syncthreads();
}

template <int M>
struct Log2 {
    static constexpr int value = 1 + Log2<M / 2>::value;
};
template <>
struct Log2<1> {
    static constexpr int value = 0;
};

// Full M-point complex FFT in LDS (natural order in and out, unnormalised).
template <typename T, int M, int NT, bool INV>
__device__ __forceinline__ void fft_lds(Cx<T> *buf, Twiddle<T> tw)
{
    constexpr int LOG = Log2<M>::value;
    int Ns = 1;
#pragma unroll
    for (int p = 0; p < LOG / 2; ++p) {
        stockham_pass<T, M, 4, NT, INV>(buf, Ns, tw);
        Ns *= 4;
    }
    if constexpr ((LOG & 1) != 0) { stockham_pass<T, M, 2, NT, INV>(buf, Ns, tw); }
}

// A value every lane holds the same copy of, moved to scalar registers
// (block-wide results read back from LDS land in vector registers).
__device__ __forceinline__ double uniform(double v)
{
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
    const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float uniform(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// ---- wave scans on DPP moves ---------------------------------------------
// v of the lane CTRL names (0 where it names none, or in rows outside
// ROWS); no LDS permute, so a step costs a few cycles instead of an LDS
// round trip.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_move(float v)
{
    return __int_as_float(dpp_move<CTRL, ROWS>(__float_as_int(v)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v)
{
    return __hiloint2double(dpp_move<CTRL, ROWS>(__double2hiint(v)), dpp_move<CTRL, ROWS>(__double2loint(v)));
}
// Inclusive sum over the lanes 0..lane of the wave: shifts by 1, 2, 4, 8
// inside rows of 16, then lane 15 of each row to the next row and lane 31 to
// the upper half.
template <typename T>
__device__ __forceinline__ T wave_scan_sum(T v)
{
    v += dpp_move<0x111, 0xf>(v);
    v += dpp_move<0x112, 0xf>(v);
    v += dpp_move<0x114, 0xf>(v);
    v += dpp_move<0x118, 0xf>(v);
    v += dpp_move<0x142, 0xa>(v);
    v += dpp_move<0x143, 0xc>(v);
    return v;
}
__device__ __forceinline__ float read_lane(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double read_lane(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Largest value of the wave (lanes that a step leaves out keep their own).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_max(float v)
{
    const int i = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float v)
{
    v = dpp_max<0x111, 0xf>(v);
    v = dpp_max<0x112, 0xf>(v);
    v = dpp_max<0x114, 0xf>(v);
    v = dpp_max<0x118, 0xf>(v);
    v = dpp_max<0x142, 0xa>(v);
    v = dpp_max<0x143, 0xc>(v);
    return read_lane(v, 63);
}
// Mean of a value per lane without the largest and the smallest of them (the
// largest when nothing is left), the same on every lane: a single outlier does
// not move it.
__device__ __forceinline__ float wave_trimmed_mean(float v)
{
    const float hi = wave_max(v), lo = -wave_max(-v);
    const bool in = !(v == hi || v == lo);
    const int n = __popcll(__ballot(in));
    const float mean = read_lane(wave_scan_sum(in ? v : 0.0f), 63) / static_cast<float>(n);
    return uniform(n > 0 ? mean : hi);
}

// ---- block reductions -------------------------------------------------
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { v += __shfl_xor(v, o, 64); }
    return v;
}
__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { v = fmax(v, __shfl_xor(v, o, 64)); }
    return v;
}

// Sum over the block; `scratch` holds NT/64 doubles.  All threads get the
// result.  Deterministic: fixed shuffle tree, then waves in order.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double *scratch)
{
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { scratch[w] = v; }
    __syncthreads();
    double s = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) { s += scratch[i]; }
    __syncthreads();
    return s;
}

template <int NT>
__device__ __forceinline__ double block_max(double v, double *scratch)
{
    v = wave_max(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { scratch[w] = v; }
    __syncthreads();
    double s = scratch[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) { s = fmax(s, scratch[i]); }
    __syncthreads();
    return s;
}

// ---- wave-level FFTs ----------------------------------------------------
// One wave (64 lanes) transforms M = 64 Q points held as Q complex values
// per lane.  Three register passes (radices R1, R2, R3, R1 R2 R3 = M) with
// two exchanges through a wave-private, padded LDS buffer; no block
// barrier is involved.  Element r of butterfly b of a pass lives in
// v[b R + r]; butterfly j = lane + 64 b reads points j + r M/R.
template <int M>
struct WavePlan;
template <>
struct WavePlan<512> {
    static constexpr int R1 = 8, R2 = 8, R3 = 8;
};
template <>
struct WavePlan<1024> {
    static constexpr int R1 = 16, R2 = 16, R3 = 4;
};
template <>
struct WavePlan<2048> {
    static constexpr int R1 = 16, R2 = 16, R3 = 8;
};

// Padded exchange index: one spare slot every 16 points breaks the
// power-of-two strides of the Stockham stores across LDS banks.
__device__ __forceinline__ int xpad(int i) { return i + (i >> 4); }
// Orders a wave's LDS stores before its later loads (LDS operations of one
// wave complete in issue order; this stops the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// Exchange addresses split into a per-lane part and a compile-time part:
// xpad(lanePart + constPart) == xpad(lanePart) + xpad(constPart) for every
// access below (one of the two parts is a multiple of 16 or their low four
// bits never carry), so each access is one base register plus an
// immediate offset.
constexpr int cpad(int i) { return i + (i >> 4); }

// cos and sin of 2 pi num / den at compile time (Taylor series around 0
// after reduction to an eighth of a turn).
constexpr double turnSeries(double x, bool sine)
{
    double term = sine ? x : 1.0, sum = term;
    for (int k = sine ? 2 : 1; k < 24; k += 2) {
        term = -term * x * x / (k * (k + 1));
        sum += term;
    }
    return sum;
}
constexpr double turnCos(int num, int den)
{
    num %= den;
    if (num < 0) { num += den; }
    if (2 * num > den) { num = den - num; }           // cos(-a) = cos(a)
    const bool neg = 4 * num > den;                   // cos(pi - a) = -cos(a)
    const int m = neg ? den - 2 * num : 2 * num;      // half turns: angle = pi m / den
    const double pi = 3.14159265358979323846;
    const double c = 4 * m <= den ? turnSeries(pi * m / den, false)
                                  : turnSeries(pi * (den - 2 * m) / (2 * den), true);
    return neg ? -c : c;
}
constexpr double turnSin(int num, int den) { return turnCos(4 * num - den, 4 * den); }

// Inter-pass twiddles of one lane's inverse transforms.  They depend on the
// lane only (not on the data or the template row), so a block computes them
// once and every transform reuses them.
//   pass 2: butterfly j has k = j mod R1 = lane mod R1 (64 is a multiple of
//           R1), the same for all of the lane's butterflies;
//   pass 3: element r of butterfly j = lane + 64 b gets W_M^-(j (r + 1/4)):
//           the transform's own twiddle W_M^-(j r) and the lane part of the
//           output weight W_{4M}^-n, n = j + m M/R3.  What is left of that
//           weight, W_{4 R3}^-m, is the same for every lane (unweight3).
// W2LDS: the pass-2 rows come from a table in LDS ((R2 - 1) R1 entries, a
// block's own; each read is a broadcast of R1 consecutive entries) instead of
// 2 (R2 - 1) registers.
// W3REG: a pass-3 row per butterfly in registers; otherwise one row for
// butterfly 0 and a constant complex product per element for the others
// (no LDS reads, and 2 (B3 - 1) R3 fewer registers).
template <typename T, int M, bool W2LDS, bool W3REG>
struct WaveTwiddles {
    using P = WavePlan<M>;
    static constexpr int NS2 = P::R1;
    static constexpr int B3 = M / (P::R3 * 64);
    static constexpr int W3 = W3REG ? B3 : 1;
    static constexpr int TABLE = W2LDS ? (P::R2 - 1) * P::R1 : 1;
    Cx<T> w2reg[W2LDS ? 1 : P::R2 - 1];
    Cx<T> w3[W3][P::R3];
    const Cx<T> *w2p;  // LDS, at the lane's entry of the first row
    // Row r of pass 2 (r = 1 .. R2 - 1).
    __device__ __forceinline__ Cx<T> w2(int r) const { return W2LDS ? w2p[(r - 1) * P::R1] : w2reg[r - 1]; }
    // The block's pass-2 table (the caller synchronises).
    __device__ __forceinline__ static void fill(Cx<T> *table, int tid, int threads, const Twiddle<T> &tw)
    {
        if constexpr (W2LDS) {
            for (int i = tid; i < TABLE; i += threads) {
                table[i] = cconj(tw((4 * M / (NS2 * P::R2)) * (i / P::R1 + 1) * (i % P::R1)));
            }
        }
    }
    __device__ __forceinline__ void init(int lane, const Twiddle<T> &tw, const Cx<T> *table)
    {
        const int k2 = lane & (NS2 - 1);
        w2p = table + k2;
        if constexpr (!W2LDS) {
            const int s2 = (4 * M / (NS2 * P::R2)) * k2;
#pragma unroll
            for (int r = 1; r < P::R2; ++r) { w2reg[r - 1] = cconj(tw(r * s2)); }
        }
#pragma unroll
        for (int b = 0; b < W3; ++b) {
#pragma unroll
            for (int r = 0; r < P::R3; ++r) { w3[b][r] = cconj(tw((lane + 64 * b) * (4 * r + 1))); }
        }
    }
};

// exp(2 pi i NUM / DEN) as a constant of type T.
template <typename T, int NUM, int DEN>
__device__ __forceinline__ Cx<T> turn()
{
    constexpr double c = turnCos(NUM, DEN), s = turnSin(NUM, DEN);
    return {static_cast<T>(c), static_cast<T>(s)};
}

// Pass 3 of an inverse transform: twiddles with the output weight, DFTs,
// and the rest of the output weight.  On return v[b R3 + m] is point
// n = lane + 64 b + m M/R3 of c_n - i c_{n+M}.
template <int B, int R, typename T, int M, typename W>
__device__ __forceinline__ void unweighted_twiddle(Cx<T> *v, const W &tw)
{
    using P = WavePlan<M>;
    if constexpr (W::W3 > 1 || B == 0) {
        v[B * P::R3 + R] = cmul(v[B * P::R3 + R], tw.w3[B][R]);
    } else {
        v[B * P::R3 + R] = cmul(v[B * P::R3 + R], cmul(tw.w3[0][R], turn<T, 16 * B * (4 * R + 1), M>()));
    }
    if constexpr (R + 1 < P::R3) {
        unweighted_twiddle<B, R + 1, T, M>(v, tw);
    } else if constexpr (B + 1 < W::B3) {
        unweighted_twiddle<B + 1, 0, T, M>(v, tw);
    }
}
template <int R, typename T, int M>
__device__ __forceinline__ void unweight3(Cx<T> *v)
{
    using P = WavePlan<M>;
    constexpr int B3 = M / (P::R3 * 64);
#pragma unroll
    for (int b = 0; b < B3; ++b) { v[b * P::R3 + R] = cmul(v[b * P::R3 + R], turn<T, R, 4 * P::R3>()); }
    if constexpr (R + 1 < P::R3) { unweight3<R + 1, T, M>(v); }
}
template <typename T, int M, typename W>
__device__ __forceinline__ void wave_pass3_inverse(Cx<T> *v, const W &tw)
{
    using P = WavePlan<M>;
    unweighted_twiddle<0, 0, T, M>(v, tw);
#pragma unroll
    for (int b = 0; b < W::B3; ++b) { mfcl::dftR<P::R3, true>(&v[b * P::R3]); }
    unweight3<1, T, M>(v);
}

// Inverse butterflies of pass 1, and of pass 2 with their twiddles.
template <typename T, int M>
__device__ __forceinline__ void wave_pass1(Cx<T> *v)
{
    constexpr int R = WavePlan<M>::R1;
#pragma unroll
    for (int b = 0; b < M / (R * 64); ++b) { mfcl::dftR<R, true>(&v[b * R]); }
}
template <typename T, int M, typename W>
__device__ __forceinline__ void wave_pass2(Cx<T> *v, const W &tw)
{
    constexpr int R = WavePlan<M>::R2, B = M / (R * 64);
#pragma unroll
    for (int r = 1; r < R; ++r) {
        const Cx<T> w = tw.w2(r);
#pragma unroll
        for (int b = 0; b < B; ++b) { v[b * R + r] = cmul(v[b * R + r], w); }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) { mfcl::dftR<R, true>(&v[b * R]); }
}

// One radix-4 pass of a 256-point forward transform held as 4 points per
// lane, and the exchange to the next pass's inputs: outputs to points
// (lane - k) 4 + k + r NS, k = lane mod NS; inputs lane + 64 r.
template <typename T, int NS, typename F>
__device__ __forceinline__ void fft256_pass(Cx<T> *y, Cx<T> *buf, int lane, F &&twiddle)
{
    const int k = lane & (NS - 1);
    if constexpr (NS > 1) {
#pragma unroll
        for (int r = 1; r < 4; ++r) { y[r] = cmul(y[r], twiddle(NS, r * k)); }
    }
    mfcl::dftR<4, false>(y);
    if constexpr (NS < 64) {
        Cx<T> *p = buf + xpad((lane - k) * 4 + k);
        const int low = ((lane - k) * 4 + k) & 15;
#pragma unroll
        for (int r = 0; r < 4; ++r) { p[r * NS + ((low + r * NS) >> 4)] = y[r]; }
        wave_lds_sync();
        const Cx<T> *q = buf + xpad(lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) { y[r] = q[cpad(64 * r)]; }
        wave_lds_sync();
    }
}

// The points X_{G k + g}, k < 256, of the forward transform of the block
// u_j = (d_j - i d_{j+M}) W_{4M}^j, M = 256 G, by one wave (residue g):
//     y_j = W_{4M}^{j (4g+1)} sum_r (d_{j+256r} - i d_{j+M+256r}) c^r,
//     c = W_{4M}^{256 (4g+1)} (its powers are table entries),  j < 256,
// then a 256-point transform of y (lane: points lane + 64 q).  The residues
// are independent, so the block's waves share one forward transform without
// a barrier inside it (it is four times shorter than on one wave while the
// others wait).  buf: 272 values of the wave's own; out[G k + g] = X.
template <typename T, int G, typename F>
__device__ __forceinline__ void forward_residue(F &&sample, int g, Cx<T> *buf, Cx<T> *out, int lane,
                                                const Twiddle<T> &tw)
{
    constexpr int M = 256 * G;
    Cx<T> y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = lane + 64 * q;
        Cx<T> s[G];
#pragma unroll
        for (int r = 0; r < G; ++r) { s[r] = {sample(j + 256 * r), -sample(j + M + 256 * r)}; }
        // the sum by halves: r and r + h with c^h, h = G/2, ..., 2, 1
#pragma unroll
        for (int h = G / 2; h >= 1; h /= 2) {
            const Cx<T> ch = tw.hi[(4 * h * (4 * g + 1)) & (16 * G - 1)];
#pragma unroll
            for (int r = 0; r < h; ++r) { s[r] = cadd(s[r], cmul(s[r + h], ch)); }
        }
        y[q] = cmul(s[0], tw(j * (4 * g + 1)));
    }
    // W_{4 NS}^e = W_{4M}^(e M / NS)
    const auto twiddle = [&](int NS, int e) { return tw(e * (M / NS)); };
    fft256_pass<T, 1>(y, buf, lane, twiddle);
    fft256_pass<T, 4>(y, buf, lane, twiddle);
    fft256_pass<T, 16>(y, buf, lane, twiddle);
    fft256_pass<T, 64>(y, buf, lane, twiddle);
#pragma unroll
    for (int r = 0; r < 4; ++r) { out[G * (lane + 64 * r) + g] = y[r]; }
}

// ---- half-size exchanges ------------------------------------------------
// The exchanges of a row transform go through a wave buffer of half the
// padded size (XHalf<M>::size), in two phases: first every value bound for
// points [0, M/2), which the lanes then load, then those bound for
// [M/2, M).  A half buffer holds point i + H M/2 at xpad(i), so the half-H
// base is buf - cpad(H M/2) and every access keeps its full-size index
// expression.  Halving the buffer is what lets more blocks share a CU's LDS.
template <int M>
struct XHalf {
    static constexpr int size = M / 2 + M / 32;
};

// Stores of a pass's outputs (radix R, butterfly phase NS) bound for half
// H.  With two or more butterflies per lane the half follows the butterfly
// index b; with one, the lane: lanes 0-31 write half 0 and 32-63 half 1.
template <typename T, int M, int R, int NS, int H>
__device__ __forceinline__ void wave_store_half(const Cx<T> *v, Cx<T> *buf, int lane)
{
    constexpr int B = M / (R * 64);
    static_assert(NS <= 64, "butterfly phase must depend on the lane only");
    const int k = lane & (NS - 1);
    Cx<T> *p = buf - cpad(H * (M / 2)) + xpad((lane - k) * R + k);
    if constexpr (B >= 2) {
#pragma unroll
        for (int b = H * (B / 2); b < (H + 1) * (B / 2); ++b) {
#pragma unroll
            for (int r = 0; r < R; ++r) { p[cpad(64 * b * R + r * NS)] = v[b * R + r]; }
        }
    } else {
        if ((lane >= 32) == (H == 1)) {
#pragma unroll
            for (int r = 0; r < R; ++r) { p[cpad(r * NS)] = v[r]; }
        }
    }
}

// Loads of the next pass's inputs (radix R) that lie in half H: input r of
// butterfly b is point lane + 64 b + r M/R, in half 0 exactly when r < R/2.
template <typename T, int M, int R, int H>
__device__ __forceinline__ void wave_load_half(Cx<T> *v, const Cx<T> *buf, int lane)
{
    constexpr int B = M / (R * 64);
    static_assert((M / R) % 16 == 0, "load offsets must be 16-aligned");
    const Cx<T> *p = buf - cpad(H * (M / 2)) + xpad(lane);
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int r = H * (R / 2); r < (H + 1) * (R / 2); ++r) { v[b * R + r] = p[cpad(64 * b + r * (M / R))]; }
    }
}

// Pass outputs in v (radix RS, phase NS) to the next pass's inputs (radix
// RL) in v, through the half buffer.
template <typename T, int M, int RS, int NS, int RL>
__device__ __forceinline__ void wave_exchange_half(Cx<T> *v, Cx<T> *buf, int lane)
{
    constexpr int Q = M / 64;
    Cx<T> u[Q];
    wave_store_half<T, M, RS, NS, 0>(v, buf, lane);
    wave_lds_sync();
    wave_load_half<T, M, RL, 0>(u, buf, lane);
    wave_lds_sync();
    wave_store_half<T, M, RS, NS, 1>(v, buf, lane);
    wave_lds_sync();
    wave_load_half<T, M, RL, 1>(u, buf, lane);
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < Q; ++i) { v[i] = u[i]; }
}

// Exchange of one component at a time through a buffer of M values of T
// (half the bytes of a complex buffer, all lanes busy, where half buffers
// with one butterfly per lane leave half the lanes idle).  One spare slot
// every 8 values: 8 consecutive values per lane then spread over the banks.
template <int M>
struct XSplit {
    static constexpr int size = M + M / 8;  // values of T
};
template <typename T, int M, int RS, int NS, int RL>
__device__ __forceinline__ void wave_exchange_split(Cx<T> *v, T *buf, int lane)
{
    static_assert(M == 64 * RS && RS == 8 && RL == 8 && (NS == 1 || NS % 8 == 0), "one radix-8 butterfly per lane");
    const int k = lane & (NS - 1);
    const int dst = (lane - k) * RS + k;
    T *p = buf + dst + (dst >> 3);
    const T *q = buf + lane + (lane >> 3);
    // value r goes to dst + r NS: the pad grows by r NS / 8 (NS = 1: not
    // within a lane's 8)
    constexpr int step = NS + NS / 8;
#pragma unroll
    for (int r = 0; r < RS; ++r) { p[r * step] = v[r].x; }
    wave_lds_sync();
    T x[RL];
#pragma unroll
    for (int r = 0; r < RL; ++r) { x[r] = q[72 * r]; }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < RS; ++r) { p[r * step] = v[r].y; }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < RL; ++r) { v[r] = {x[r], q[72 * r]}; }
    wave_lds_sync();
}
// wave_passes12_half one component at a time.
template <typename T, int M, typename W>
__device__ __forceinline__ void wave_passes12_split(Cx<T> *v, T *buf, int lane, const W &tw)
{
    using P = WavePlan<M>;
    wave_pass1<T, M>(v);
    wave_exchange_split<T, M, P::R1, 1, P::R2>(v, buf, lane);
    wave_pass2<T, M>(v, tw);
    wave_exchange_split<T, M, P::R2, P::R1, P::R3>(v, buf, lane);
}

// Inverse passes 1 and 2 on data in registers (v[b R1 + r] = point lane +
// 64 b + r M/R1), up to the inputs of pass 3, through a half buffer.
template <typename T, int M, typename W>
__device__ __forceinline__ void wave_passes12_half(Cx<T> *v, Cx<T> *buf, int lane, const W &tw)
{
    using P = WavePlan<M>;
    wave_pass1<T, M>(v);
    wave_exchange_half<T, M, P::R1, 1, P::R2>(v, buf, lane);
    wave_pass2<T, M>(v, tw);
    wave_exchange_half<T, M, P::R2, P::R1, P::R3>(v, buf, lane);
}

// True when the Lt samples of the window at i are all equal (its exact
// value is then 0: zero numerator over the floor of the norm), from the
// equal-neighbour bits.
__device__ __forceinline__ bool constant_window(const unsigned *eqw, int i, int Lt)
{
    const int end = i + Lt - 1;  // bits [i, end)
    for (int p = i; p < end;) {
        const int b = p & 31;
        const int take = min(32 - b, end - p);
        const unsigned mask = (take == 32 ? ~0u : ((1u << take) - 1u)) << b;
        if ((eqw[p >> 5] & mask) != mask) { return false; }
        p += take;
    }
    return true;
}

}  // namespace mfdev
