// Time-domain correlation of short templates on MFMA (the optional
// short-template path; no FFT).
//
// For one lane (a channel and its rows, every template at most KT taps)
// the numerators form a Hankel-by-template GEMM
//     D[j][i] = sum_k t~_j[k] * x~[i + k],
// t~_j the demeaned unit-norm template j (zero past its length) and
// x~ = (x - a) / s the block's samples with the block anchor a removed and
// scaled by their RMS s.  Both operands are split into 16-bit parts:
//  - FP16 (11-bit significand): hi = round(v), lo = round(v - hi); the
//    products hi*hi, hi*lo and lo*hi;
//  - BF16 (8-bit significand): hi, mid = round(v - hi),
//    lo = round(v - hi - mid); the six products hi*hi, hi*mid, mid*hi,
//    hi*lo, lo*hi and mid*mid (the dropped ones, mid*lo, lo*mid and lo*lo,
//    are below 2^-24 of |t||x|).
// v_mfma_f32_16x16x32 accumulates them in FP32: hi*hi in its own
// accumulator, the smaller products in a second one.
// rho = s * D * scale with the window normalisation from FP64 prefix sums
// of the block.
//
// Work item: IS = 512 consecutive outputs of the lane and up to 192 rows.
// Each of the 4 waves takes 16 rows at a time: their split taps stay in
// registers (weight-stationary, parts * KT / 8 VGPRs) while the wave walks
// the 32 output tiles of 16; the Hankel operand's entry p, the 8 samples
// x~[p .. p+7], is read from LDS for one k-step of 32 per tile and part and
// stays in a ring of registers.
//
// Accuracy: per window |d rho| <= eps_m * sqrt(Lt S2) / den with
// eps_m = eps_split + (4 sqrt(KT/16) + 4) 2^-24 (FP32 accumulation over at
// most KT / 16 accumulator updates -- the kernel makes KT / 32 -- and the
// FP32 epilogue on the FP64 window sums), S2 the
// window's sum of (x - a)^2 and den its centred norm; eps_split is the
// relative size of the dropped products and split residuals: 3 * 2^-22 for
// the FP16 pair (3 u^2, u = 2^-11) and 3 * 2^-24 for the BF16 triple
// (3 u^3, u = 2^-8); the FP16 pair also loses low parts below its smallest
// subnormal, at most 2^-25 of the block's RMS per sample.  Windows whose
// bound exceeds the FP32 tolerance get their numerator recomputed in FP64
// from the anchored samples (the window norm from the prefix sums is accurate
// there); windows whose FP64 variance lost too many digits get the exact
// two-pass Pearson value, as in the FFT path.
#include "mf_device.hpp"
#include "mf_kernels.hpp"
#include <cfloat>

using namespace mfdev;

namespace mfk {

namespace {

constexpr int NT = kThreads;
constexpr int IS = kTdOutputsPerItem;  // outputs per work item

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

// The 16-bit operand type's parts and its v_mfma_f32_16x16x32 form.
template <typename MT>
struct TdTraits;
template <>
struct TdTraits<_Float16> {
    using vec8 = f16x8;
    static constexpr int parts = 2;
    __device__ static f32x4 mfma(vec8 a, vec8 b, f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <>
struct TdTraits<__bf16> {
    using vec8 = bf16x8;
    static constexpr int parts = 3;
    __device__ static f32x4 mfma(vec8 a, vec8 b, f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

constexpr int kTdCoopFlags = 4;  // at most this many left at the end: the wave shares each window

// Tiles with at least this many windows whose numerator is recomputed take
// the whole tile's numerators on FP64 MFMA (16 x 16 windows, 64 products of
// 64 cycles at 256 taps: 4100 cycles of one SIMD), fewer go one by one to
// the queue kernel (227 SIMD cycles each, measured: 10.7 M windows of about
// 190 taps in 0.99 ms): the lines cross at 18.
constexpr int kTdTileFlags = 20;
static_assert(kTdTileFlags > 16, "the host counts no tiles of a group of one row");

// A window's norm is taken from the block's prefix sums when its den2 is above
// kTdCancel Lt E (E the block's sum of d^2).  A prefix sum carries at most 14
// roundings of values up to E (three samples of a thread, the wave's scan, the
// waves before), so S2, a difference of two, is within 28 x 2^-53 E = 3.1e-15 E
// and den2 within 3.1e-15 Lt E: 1.6e-6 of rho at this line.  Windows 90 dB below
// their block take the two-pass value instead (|rho| 0.9 beside a spike of 1e7
// times the noise was off by 1.6e-5 with a line of 1e-12).
constexpr double kTdCancel = 1.0e-9;

// FP64 prefix sums of d = x - a and of d^2 at one sample.
struct __align__(16) TdSums {
    double s1, s2;
};

// Exact FP64 value of one flagged window at item offset i, over taps
// m = m0, m0 + step, ... (one lane: 0, 1; a whole wave: lane, 64, summed
// across the wave).
//  - cancelled variance (canc): one pass over d = x - x0, x0 the window's
//    first sample (every d is exact in FP64), giving
//    rho = sum t d / sqrt(sum d^2 - (sum d)^2 / Lt); the template has zero
//    mean, so sum t d is the centred numerator, and with the shift inside
//    the window the variance keeps its digits (a constant window gives 0);
//  - noise flag: the numerator sum t (x - a) from the anchored samples with
//    the window norm from the block's FP64 prefix sums, accurate there.
// |rho| > 1.1 gives 0 (the reference's tooBig rule).
__device__ double exact_window_td(const float *raw, const TdSums *P, int i,
                                  gptr<const double> t, int Lt, double a, bool canc, int m0, int step)
{
    const double shift = canc ? static_cast<double>(raw[i]) : a;
    double s1 = 0, s2 = 0, dn = 0;
#pragma unroll 8
    for (int m = m0; m < Lt; m += step) {
        const double d = static_cast<double>(raw[i + m]) - shift;
        s1 += d;
        s2 = fma(d, d, s2);
        dn = fma(t[m], d, dn);
    }
    if (step > 1) {
        s1 = wave_sum(s1);
        s2 = wave_sum(s2);
        dn = wave_sum(dn);
    }
    double rho;
    if (canc) {
        rho = dn / fmax(DBL_EPSILON, sqrt(fmax(0.0, s2 - s1 * s1 / Lt)));
    } else {
        const double S1 = P[i + Lt].s1 - P[i].s1;
        const double den2 = Lt * (P[i + Lt].s2 - P[i].s2) - S1 * S1;
        rho = dn * sqrt(Lt / den2);
    }
    return fabs(rho) > 1.1 ? 0.0 : rho;
}

// One work item's staged samples in LDS, shared by both tile shapes.
template <typename MT, int KT>
struct TdStage {
    static constexpr int NP = TdTraits<MT>::parts;
    static constexpr int SPAN = IS + KT;  // samples one item reads
    // x~ of each part as pairs of samples in two copies: pair w of copy c is
    // samples 2 w + c and 2 w + c + 1, so the 8 samples from p on are four
    // consecutive words of copy p mod 2
    unsigned x2[NP][2][SPAN / 2];
    float raw[SPAN];                      // samples (FP32), for exact windows
    TdSums P[SPAN + 1];                   // prefix sums
    double tot1[NT / 64], tot2[NT / 64];
    unsigned eqw[(SPAN + 31) / 32];       // bit p: sample p equals sample p + 1
    unsigned short run[SPAN];             // set bits from bit p on, up to 256 (blocks with any):
                                          // the window at p is constant when run[p] >= Lt - 1
};

// What the epilogue needs of the staged block: the anchor a, the scale s
// of x~ (FP32) and the cancellation floor kTdCancel E (per tap of Lt).
struct TdBlock {
    double a;
    float scF;
    float flK;
    bool equal;  // some sample equals its neighbour: `run` is filled
};

// Stages outputs [base, base + IS) of lane sg: loads the samples, takes the
// anchor (a mean of 64 samples spread over the block, taken by every wave: any
// value near the samples will do; without the largest and the smallest, as a
// glitch of 100 times the noise among them moved it far enough to make every
// window of the item noisy) and the RMS about it, splits x~ into
// its parts, builds the FP64 prefix sums and the equal-neighbour bits.  Each
// thread takes consecutive samples and the scan runs on DPP moves, with one
// barrier inside (the split by LDS copies of every entry, sums behind four
// barriers and bits on one wave took 20 % of the kernel).  Ends with the
// block synchronised.
template <typename MT, int KT>
__device__ __forceinline__ TdBlock td_stage(TdStage<MT, KT> &sm, const Seg &sg, long long base)
{
    constexpr int NP = TdTraits<MT>::parts;
    constexpr int SPAN = TdStage<MT, KT>::SPAN;
    constexpr int SPT = (SPAN + NT - 1) / NT;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    // 1. samples, anchor, running sums
    const gptr<const float> x = to_global(static_cast<const float *>(sg.x)) + base;
    const int nSamp = static_cast<int>(min(static_cast<long long>(SPAN), sg.n - base));
    const float spread = x[(lane * nSamp) >> 6];
    const int p0 = tid * SPT;
    float v[SPT];
#pragma unroll
    for (int q = 0; q < SPT; ++q) { v[q] = p0 + q < nSamp ? x[p0 + q] : 0.0f; }
    const float after = p0 + SPT < nSamp ? x[p0 + SPT] : 0.0f;
    if (tid < (SPAN + 31) / 32) { sm.eqw[tid] = 0u; }
    const double a = static_cast<double>(wave_trimmed_mean(spread));
    double t1 = 0, t2 = 0;
    double l1[SPT], l2[SPT];  // exclusive sums inside the thread
#pragma unroll
    for (int q = 0; q < SPT; ++q) {
        const double d = p0 + q < nSamp ? static_cast<double>(v[q]) - a : 0.0;
        l1[q] = t1;
        l2[q] = t2;
        t1 += d;
        t2 += d * d;
        if (p0 + q < SPAN) { sm.raw[p0 + q] = v[q]; }
    }
    const double i1 = wave_scan_sum(t1), i2 = wave_scan_sum(t2);
    if (lane == 63) {
        sm.tot1[wave] = i1;
        sm.tot2[wave] = i2;
    }
    __syncthreads();
    double energy = 0, o1 = 0, o2 = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        if (w == wave) {
            o1 += i1 - t1;
            o2 = energy + (i2 - t2);
        } else if (w < wave) {
            o1 += sm.tot1[w];
        }
        energy += sm.tot2[w];
    }
    // 2. prefix sums P[p] = sum over q < p, equal-neighbour bits
    int equal = 0;
#pragma unroll
    for (int q = 0; q < SPT; ++q) {
        if (p0 + q < SPAN) { sm.P[p0 + q] = TdSums{o1 + l1[q], o2 + l2[q]}; }
        if (p0 + q == SPAN - 1) {
            const double d = p0 + q < nSamp ? static_cast<double>(v[q]) - a : 0.0;
            sm.P[SPAN] = TdSums{o1 + l1[q] + d, o2 + l2[q] + d * d};
        }
        const float next = q + 1 < SPT ? v[q + 1 < SPT ? q + 1 : q] : after;
        if (p0 + q + 1 < SPAN && v[q] == next) {
            atomicOr(&sm.eqw[(p0 + q) >> 5], 1u << ((p0 + q) & 31));
            equal = 1;
        }
    }
    // 3. the parts of x~ = (x - a) / sc.  The FP32 value is the sum of its
    //    parts exactly (each remainder is exact in FP32 and the parts
    //    together hold at least 24 significant bits).
    const double sc = energy > 0 ? sqrt(energy / nSamp) : 1.0;
    const float inv = static_cast<float>(1.0 / sc);
#pragma unroll
    for (int q = 0; q < SPT; ++q) {
        const int p = p0 + q;
        if (p < SPAN) {
            float rest = p < nSamp ? static_cast<float>((static_cast<double>(v[q]) - a) * inv) : 0.0f;
#pragma unroll
            for (int pt = 0; pt < NP; ++pt) {
                const MT part = static_cast<MT>(rest);
                rest -= static_cast<float>(part);
                reinterpret_cast<MT *>(sm.x2[pt][0])[p] = part;
                if (p > 0) { reinterpret_cast<MT *>(sm.x2[pt][1])[p - 1] = part; }
                if (p == SPAN - 1) { reinterpret_cast<MT *>(sm.x2[pt][1])[p] = static_cast<MT>(0.0f); }
            }
        }
    }
    const bool any = __syncthreads_or(equal) != 0;
    if (any) {  // 4. run lengths of the bits
        constexpr int W = (SPAN + 31) / 32;
        int run = 0;
        for (int p = p0 + SPT; run < 256 && p < SPAN;) {  // of the next thread's first sample
            const unsigned rest = sm.eqw[p >> 5] >> (p & 31);
            const int take = min(32 - (p & 31), SPAN - p);
            const int ones = min(rest == ~0u ? 32 : __ffs(~rest) - 1, take);
            run += ones;
            if (ones < take) { break; }
            p += take;
        }
        static_assert(W * 32 >= SPAN, "words");
#pragma unroll
        for (int q = SPT - 1; q >= 0; --q) {
            const int p = p0 + q;
            if (p < SPAN) {
                run = (sm.eqw[p >> 5] >> (p & 31)) & 1u ? min(run + 1, 256) : 0;
                sm.run[p] = static_cast<unsigned short>(run);
            }
        }
        __syncthreads();
    }
    return TdBlock{a, static_cast<float>(sc), static_cast<float>(kTdCancel * energy), any};
}

// A dead lane's item: zeros in every row.
__device__ __forceinline__ void td_dead(const TdItem &item, const TdRow *__restrict__ rows)
{
    const long long base = item.seg0;
    for (int r = 0; r < item.nRows; ++r) {
        const TdRow row = rows[item.rowBegin + r];
        const int nv = static_cast<int>(min(static_cast<long long>(IS), row.nOut - base));
        gptr<float> out = to_global(static_cast<float *>(row.out)) + base;
        for (int i = threadIdx.x; i < nv; i += NT) { out[i] = 0.0f; }
    }
}

// Tiles of 16 rows x 16 outputs on v_mfma_f32_16x16x32: each wave holds the
// split taps of 16 rows (parts * KT / 8 VGPRs: 96 for the BF16 triple at
// KT = 256; tiles of 32 rows would need 192 and leave one wave per SIMD)
// and walks the item's 32 output tiles; the 4 waves take 64 rows at a
// time, in up to three row groups.  A lane holds column
// i = lane % 16 and rows 4 (lane / 16) + r, r = 0..3: their epilogue
// constants stay in registers for the row group, and each quarter wave
// stores 16 consecutive outputs of its row.
constexpr int kTdTiles = IS / 16;        // output tiles of 16 per item
constexpr int kTdRingParts = 2;          // operand parts whose steps stay in registers
constexpr int kTdFixList = 64 + 4 * 64;  // carried over plus one tile's windows

// Blocks per CU the register budget is capped for: two, at KT = 256 64 (FP16
// pair) or 96 (BF16 triple) registers of taps and 64 of the operand ring.
constexpr int kTdBlocks = 2;

template <typename MT, int KT>
__global__ __launch_bounds__(NT, kTdBlocks) void tdcorr_kernel(const TdItem *__restrict__ items,
                                                       const Seg *__restrict__ segs,
                                                       const TdRow *__restrict__ rows, FixQueue queue)
{
    using Tr = TdTraits<MT>;
    using V8 = typename Tr::vec8;
    typedef int WordsU __attribute__((ext_vector_type(4), aligned(4)));  // four words at any word
    constexpr int NP = Tr::parts;
    constexpr int NS = KT / 32;  // k-steps of 32
    constexpr int RP = kTdRingParts;
    __shared__ __align__(16) TdStage<MT, KT> sm;
    // flagged windows of each wave's tiles: bit r flags the lane's window
    // r, bit 4 + r marks a cancelled variance
    __shared__ unsigned char fq[NT / 64][kTdTiles][64];
    // each wave's list of flagged windows to recompute when the device
    // queue is full
    __shared__ unsigned short fixList[NT / 64][kTdFixList];

    const TdItem item = items[blockIdx.x];
    const Seg sg = segs[item.seg];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int quad = lane >> 4;  // k-group of the operands, row group of the result
    // The taps of k-group quad: 8 kq + 0..7 of each k-step of 32, with kq =
    // 0, 2, 1, 3 for quad = 0..3 (A and B alike, so the products summed are
    // the same): each half wave then reads 32 consecutive Hankel entries
    // (quads 0 and 1: i0 + 0..31; 2 and 3: i0 + 8..39) instead of two
    // overlapping runs of 16 in the same LDS banks.
    const int kq = ((quad & 1) << 1) | (quad >> 1);
    const int c16 = lane & 15;   // output column
    const long long base = item.seg0;

    if (sg.dead) {
        td_dead(item, rows);
        return;
    }
    const TdBlock blk = td_stage(sm, sg, base);
    const double a = blk.a;
    const float scF = blk.scF;
    const float flK = blk.flK;

    constexpr float kUnder = NP == 2 ? static_cast<float>(2.98023223876953125e-08 / kTdRhoTol) : 0.0f;
    unsigned long long nFlag = 0, nCanc = 0;  // windows recomputed by this wave, in full
    for (int g = 0; 64 * g < item.nRows; ++g) {
        const int rowBase = item.rowBegin + 64 * g + 16 * wave;
        const int nMine = min(16, item.nRows - 64 * g - 16 * wave);
        if (nMine <= 0) { break; }
        // split taps (A operand: row = lane % 16, taps 32 s + 8 kq + 0..7
        // of each part)
        V8 ap[NP][NS];
        {
            const bool has = c16 < nMine;
            const MT *f = has ? static_cast<const MT *>(rows[rowBase + c16].frag) : nullptr;
#pragma unroll
            for (int pt = 0; pt < NP; ++pt) {
#pragma unroll
                for (int st = 0; st < NS; ++st) {
                    if (has) {
                        const gptr<const i32x4> fh = to_global(reinterpret_cast<const i32x4 *>(f));
                        ap[pt][st] = __builtin_bit_cast(V8, fh[pt * (KT / 8) + 4 * st + kq]);
                    } else {
                        ap[pt][st] = __builtin_bit_cast(V8, i32x4{0, 0, 0, 0});
                    }
                }
            }
        }
        // the epilogue constants of the lane's 4 rows (absent rows: no
        // outputs, and a length that keeps the prefix reads in the span)
        int LtR[4], nvR[4];
        float kcR[4], knR[4], slR[4], floorF[4];
        gptr<float> outR[4];
        int fullOut = IS;  // outputs every row of the group has
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 4 * quad + r;
            if (j < nMine) {
                const TdRow row = rows[rowBase + j];
                LtR[r] = row.Lt;
                nvR[r] = static_cast<int>(max(0ll, min(static_cast<long long>(IS), row.nOut - base)));
                kcR[r] = row.kc;
                knR[r] = row.kn;
                slR[r] = row.sqrtLt * scF;
                outR[r] = to_global(static_cast<float *>(row.out)) + base;
            } else {
                LtR[r] = 1;
                nvR[r] = 0;
                kcR[r] = 0.0f;
                knR[r] = 0.0f;
                slR[r] = 0.0f;
                outR[r] = nullptr;
            }
            // below the cancellation floor, or (FP16) so quiet beside the
            // block's RMS s that the samples' low parts underflow: their
            // rounding, 2^-25 s each, is sqrt(Lt) 2^-25 s in the numerator
            const float under = kUnder * scF * static_cast<float>(LtR[r]);
            floorF[r] = fmaf(under, under, flK * static_cast<float>(LtR[r]));
            // An absent row flags nothing: its one-sample windows have no norm,
            // and with the block's floor every tile of a group of fewer than 16
            // rows took the branch for flagged windows.
            if (j >= nMine) { floorF[r] = -INFINITY; }
            fullOut = min(fullOut, nvR[r]);
        }
        fullOut = min(fullOut, __shfl_xor(fullOut, 16, 64));
        fullOut = __builtin_amdgcn_readfirstlane(min(fullOut, __shfl_xor(fullOut, 32, 64)));
        unsigned tiles = 0;  // tiles with flagged windows (wave-uniform)
        // B operand: column i0 + c16, taps 32 st + 8 kq + 0..7 = entry
        // i0 + c16 + 8 kq + 32 st.  Step st of the tile 32 outputs on is this
        // tile's step st + 1, so the wave walks the even tiles, then the odd
        // ones, with its steps in a ring of registers and reads one new step
        // per tile.  (With every step read for every tile the LDS pipe, shared
        // by the four SIMDs, set the time: 168 of its cycles per tile against
        // 384 / 4 of the matrix cores.)  The ring turns with the unrolled
        // tiles, so its slots are compile-time.
        for (int par = 0; par < 2; ++par) {
            const int e0 = 16 * par + c16 + 8 * kq;
            const auto entry = [&](int pt, int step) {
                return __builtin_bit_cast(V8, *reinterpret_cast<const WordsU *>(&sm.x2[pt][e0 & 1][(e0 >> 1) + 16 * step]));
            };
            V8 ring[RP][NS];
#pragma unroll
            for (int pt = 0; pt < RP; ++pt) {
#pragma unroll
                for (int st = 0; st < NS; ++st) { ring[pt][st] = entry(pt, st); }
            }
            for (int t0 = 0; t0 < kTdTiles / 2; t0 += NS) {
#pragma unroll
                for (int u = 0; u < NS; ++u) {
                    const int t = t0 + u;
                    const int tile = 2 * t + par;
                    const int i0 = 16 * tile;
                    f32x4 acc0 = {}, acc1 = {}, acc2 = {};
#pragma unroll
                    for (int st = 0; st < NS; ++st) {
                        const V8 b0 = ring[0][(u + st) % NS], b1 = ring[1][(u + st) % NS];
                        acc0 = Tr::mfma(ap[0][st], b0, acc0);
                        acc1 = Tr::mfma(ap[0][st], b1, acc1);
                        acc2 = Tr::mfma(ap[1][st], b0, acc2);
                        if constexpr (NP == 3) {
                            const V8 b2 = entry(NP - 1, t + st);  // the BF16 triple's third part
                            acc1 = Tr::mfma(ap[0][st], b2, acc1);
                            acc2 = Tr::mfma(ap[NP - 1][st], b0, acc2);
                            acc1 = Tr::mfma(ap[1][st], b1, acc1);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) { acc1[r] += acc2[r]; }
                    // the next tile's last step (the last tile reads its own again)
                    const int next = min(t + 1, kTdTiles / 2 - 1) + NS - 1;
#pragma unroll
                    for (int pt = 0; pt < RP; ++pt) { ring[pt][u] = entry(pt, next); }
                    // epilogue: normalise, flag, store.  A window is flagged unless
                    // den2 - kn S2 is above the cancellation floor (kc is far below
                    // kn, so its test is left to the windows this one flags); where
                    // every row has the tile's outputs, flagged ones are stored too
                    // and overwritten later.
                    const int i = i0 + c16;
                    const TdSums pi = sm.P[i];
                    const bool full = i0 + 16 <= fullOut;  // uniform
                    float rho[4];
                    unsigned long long flags[4], any = 0;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        // window sums in FP64 (differences of the block's prefix
                        // sums), the rest in FP32
                        const TdSums pe = sm.P[i + LtR[r]];
                        const double S1 = pe.s1 - pi.s1, S2 = pe.s2 - pi.s2;
                        const float d2 = static_cast<float>(fma(-S1, S1, LtR[r] * S2));
                        flags[r] = __ballot(!(fmaf(-knR[r], static_cast<float>(S2), d2) > floorF[r]));
                        any |= flags[r];
                        float y = __builtin_amdgcn_rsqf(d2);
                        y = y * (1.5f - 0.5f * d2 * y * y);
                        rho[r] = (acc0[r] + acc1[r]) * (slR[r] * y);
                    }
                    if (full) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) { outR[r][i] = rho[r]; }
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (i < nvR[r]) { outR[r][i] = rho[r]; }
                        }
                    }
                    if (any != 0ull) {
                        // exactly constant windows (a gap's) are 0 at once; the rest
                        // wait for the end of the row group
                        const int run = blk.equal ? sm.run[i] : 0;
                        unsigned bits = 0;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const bool flag = i < nvR[r] && ((flags[r] >> lane) & 1u);
                            const bool flat = flag && run >= LtR[r] - 1;  // a one-sample window always
                            if (flat) { outR[r][i] = 0.0f; }
                            const unsigned nFlat = static_cast<unsigned>(__popcll(__ballot(flat)));
                            nFlag += nFlat;
                            nCanc += nFlat;
                            bits |= (flag && !flat ? 1u : 0u) << r;
                        }
                        if (__ballot(bits != 0u) != 0ull) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const TdSums pe = sm.P[i + LtR[r]];
                                const double S1 = pe.s1 - pi.s1, S2 = pe.s2 - pi.s2;
                                const float d2 = static_cast<float>(fma(-S1, S1, LtR[r] * S2));
                                const float floorR = fmaf(kcR[r], static_cast<float>(S2), flK * static_cast<float>(LtR[r]));
                                bits |= (((bits >> r) & 1u) && !(d2 > floorR) ? 1u : 0u) << (4 + r);
                            }
                        }
                        if (__ballot(bits != 0u) != 0ull) {
                            fq[wave][tile][lane] = static_cast<unsigned char>(bits);
                            tiles |= 1u << tile;
                        }
                    }
                }
            }
        }
        // flagged windows of the row group, after its tile loop: a tile of
        // many windows that keep their norm is recorded for the tile launch
        // (numerators on FP64 MFMA); the others go to the device queue
        // (fix_kernel recomputes them after the launch), or, when it
        // is full, to the wave's list, recomputed here one window per lane
        // in passes of 64 (a few left at the end: the whole wave on one
        // window at a time).  List entry: tile (5 bits), step r (2 bits),
        // lane (6 bits), cancelled (1 bit).
        unsigned short *list = fixList[wave];
        int nList = 0;  // wave-uniform
        auto entryWindow = [&](unsigned e, int &wi, TdRow &row, bool &cr) {
            const int t = (e >> 8) & 31, r = (e >> 6) & 3, l = e & 63;
            wi = 16 * t + (l & 15);
            row = rows[rowBase + 4 * (l >> 4) + r];
            cr = (e >> 13) & 1u;
        };
        auto runList = [&](bool all) {
            int done = 0;
            while (nList - done >= 64 || (all && nList - done > kTdCoopFlags)) {
                const int n = min(64, nList - done);
                if (lane < n) {
                    int wi;
                    TdRow row;
                    bool cr;
                    entryWindow(list[done + lane], wi, row, cr);
                    const double rho =
                        exact_window_td(sm.raw, sm.P, wi, to_global(row.tmpl), row.Lt, a, cr, 0, 1);
                    to_global(static_cast<float *>(row.out))[base + wi] = static_cast<float>(rho);
                }
                done += n;
            }
            if (all) {
                for (; done < nList; ++done) {
                    int wi;
                    TdRow row;
                    bool cr;
                    entryWindow(list[done], wi, row, cr);  // uniform entry: the wave shares it
                    const double rho =
                        exact_window_td(sm.raw, sm.P, wi, to_global(row.tmpl), row.Lt, a, cr, lane, 64);
                    if (lane == 0) { to_global(static_cast<float *>(row.out))[base + wi] = static_cast<float>(rho); }
                }
            } else if (done > 0) {
                // the remainder (under 64 entries) moves to the front: every
                // lane reads before any lane writes (one instruction each)
                const int rest = nList - done;
                const unsigned short v = lane < rest ? list[done + lane] : 0;
                if (lane < rest) { list[lane] = v; }
            }
            nList -= done;
        };
        while (tiles != 0u) {
            const int tile = __ffs(tiles) - 1;
            tiles &= tiles - 1u;
            const int i = 16 * tile + c16;
            const unsigned word = fq[wave][tile][lane];
            const unsigned flg = word & 15u;
            const unsigned cnc = word >> 4;
            unsigned keep = flg;  // the window queue's
            const unsigned noisy = flg & ~cnc;
            int n = 0, nNoisy = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                n += __popcll(__ballot((flg >> r) & 1u));
                nNoisy += __popcll(__ballot((noisy >> r) & 1u));
            }
            nFlag += static_cast<unsigned>(n);
            nCanc += static_cast<unsigned>(n - nNoisy);
            if (nNoisy >= kTdTileFlags) {  // the tile launch's, marked by NaN
                if (lane == 0) {
                    // the list has a record for every tile of the launch
                    gptr<int> rec = to_global(queue.over) + 4 * atomicAdd(queue.overCount, 1ull);
                    rec[0] = rowBase;
                    rec[1] = nMine;
                    rec[2] = static_cast<int>(base) + 16 * tile;
                    rec[3] = __float_as_int(static_cast<float>(a));  // a is an FP32 value
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if ((noisy >> r) & 1u) { outR[r][i] = __builtin_nanf(""); }
                }
                keep &= cnc;
                n -= nNoisy;
            }
            if (n == 0) { continue; }
            unsigned long long q0 = 0;
            if (lane == 0) { q0 = atomicAdd(queue.count, static_cast<unsigned long long>(n)); }
            q0 = __shfl(q0, 0, 64);
            if (q0 <= queue.cap && static_cast<unsigned long long>(n) <= queue.cap - q0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool mine = (keep >> r) & 1u;
                    const unsigned long long bal = __ballot(mine);
                    if (mine) {
                        const unsigned long long at = q0 + __popcll(bal & ((1ull << lane) - 1ull));
                        const unsigned rowCode =
                            static_cast<unsigned>(rowBase + 4 * quad + r) | (((cnc >> r) & 1u) << 31);
                        gptr<unsigned long long> e = to_global(reinterpret_cast<unsigned long long *>(queue.entries));
                        e[at] = (static_cast<unsigned long long>(base + i) << 32) | rowCode;
                    }
                    q0 += __popcll(bal);
                }
                continue;
            }
            // The queue is full.  A reservation that straddles its end
            // leaves the slots [q0, cap) unused: they get the empty entry,
            // which fix_kernel skips (it reads min(count, cap) entries).
            if (q0 < queue.cap) {
                gptr<unsigned long long> e = to_global(reinterpret_cast<unsigned long long *>(queue.entries));
                for (unsigned long long k = q0 + lane; k < queue.cap; k += 64) { e[k] = kFixEmpty; }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool mine = (keep >> r) & 1u;
                const unsigned long long bal = __ballot(mine);
                if (mine) {
                    const int at = nList + __popcll(bal & ((1ull << lane) - 1ull));
                    list[at] = static_cast<unsigned short>((tile << 8) | (r << 6) | lane | (((cnc >> r) & 1u) << 13));
                }
                nList += __popcll(bal);
            }
            runList(false);
        }
        runList(true);
    }
    if (sg.flagged != nullptr && nFlag != 0ull && lane == 0) {
        atomicAdd(sg.flagged, nFlag);
        if (nCanc != 0ull) { atomicAdd(sg.flagged + 1, nCanc); }
    }
}

// The recorded tiles of a time-domain launch, one wave each: the windows
// marked NaN among 16 rows x 16 outputs are recomputed in FP64, numerators on
// v_mfma_f64_16x16x4 and norms from prefix sums of the tile's own samples,
// about the anchor of the item that recorded them.  Their energy about it is
// at most the item's, so the item's cancellation test holds for these sums
// too; about a sample of the tile's own, which may be a spike or the end of a
// loud stretch, it would not.  A launch of its own because a gap's edge flags
// every tile of a few items: recomputed inside them, those items ran three
// to four times longer than the rest and the chip waited for them (0.8 of
// 2.84 ms, 256 rows x 4 channels x 1 M samples).
constexpr int kTileSpan = 320;  // samples a tile may read (16 + 255), five per lane
__global__ __launch_bounds__(NT) void fix_tiles_kernel(const TdRow *__restrict__ rows, FixQueue queue)
{
    constexpr int PER = kTileSpan / 64;
    __shared__ float rawS[NT / 64][kTileSpan];
    __shared__ TdSums sumS[NT / 64][kTileSpan + 1];
    const unsigned long long n = *queue.overCount;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, quad = lane >> 4, c16 = lane & 15;
    float *raw = rawS[wave];
    TdSums *P = sumS[wave];
    for (unsigned long long k = static_cast<unsigned long long>(blockIdx.x) * (NT / 64) + wave; k < n;
         k += static_cast<unsigned long long>(gridDim.x) * (NT / 64)) {
        const gptr<const int> rec = to_global(static_cast<const int *>(queue.over)) + 4 * k;
        const int rowBase = __builtin_amdgcn_readfirstlane(rec[0]);
        const int nMine = __builtin_amdgcn_readfirstlane(rec[1]);
        const int pos = __builtin_amdgcn_readfirstlane(rec[2]);
        const TdRow mine = rows[rowBase + min(c16, nMine - 1)];
        const gptr<const double> t = to_global(mine.tmpl);
        const int LtA = c16 < nMine ? mine.Lt : 0;
        // the longest row, and the samples from pos on that the windows reach:
        // no others, whose value (a NaN, a spike) the item's test has not seen
        int LtMax = mine.Lt, reach = static_cast<int>(min(mine.nOut - pos, 16ll)) + mine.Lt - 1;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            LtMax = max(LtMax, __shfl_xor(LtMax, o, 64));
            reach = max(reach, __shfl_xor(reach, o, 64));
        }
        LtMax = __builtin_amdgcn_readfirstlane(LtMax);
        const gptr<const float> x = to_global(mine.x) + pos;
        const double a = static_cast<double>(__int_as_float(__builtin_amdgcn_readfirstlane(rec[3])));
        float v[PER];
        double l1[PER], l2[PER], t1 = 0, t2 = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int j = lane * PER + q;
            v[q] = j < reach ? x[j] : 0.0f;
            const double d = j < reach ? static_cast<double>(v[q]) - a : 0.0;
            l1[q] = t1;
            l2[q] = t2;
            t1 += d;
            t2 += d * d;
        }
        const double e1 = wave_scan_sum(t1) - t1, e2 = wave_scan_sum(t2) - t2;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            raw[lane * PER + q] = v[q];
            P[lane * PER + q] = TdSums{e1 + l1[q], e2 + l2[q]};
        }
        if (lane == 63) { P[kTileSpan] = TdSums{e1 + t1, e2 + t2}; }
        wave_lds_sync();
        f64x4 acc = {};
        double tk[4];
        const auto taps = [&](int k0) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int m = k0 + 4 * u + quad;
                tk[u] = m < LtA ? t[m] : 0.0;
            }
        };
        taps(0);
        for (int k0 = 0; k0 < LtMax; k0 += 16) {
            double tc[4], dk[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                tc[u] = tk[u];
                dk[u] = static_cast<double>(raw[c16 + k0 + 4 * u + quad]) - a;
            }
            taps(k0 + 16);  // in flight through this step's products
#pragma unroll
            for (int u = 0; u < 4; ++u) { acc = __builtin_amdgcn_mfma_f64_16x16x4f64(tc[u], dk[u], acc, 0, 0, 0); }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 4 * r + quad;  // the result's row
            if (j < nMine) {
                const TdRow row = rows[rowBase + j];
                if (static_cast<long long>(pos) + c16 < row.nOut) {
                    gptr<float> out = to_global(static_cast<float *>(row.out)) + pos + c16;
                    if (isnan(*out)) {
                        const double S1 = P[c16 + row.Lt].s1 - P[c16].s1;
                        const double den2 = row.Lt * (P[c16 + row.Lt].s2 - P[c16].s2) - S1 * S1;
                        double rho = acc[r] * sqrt(row.Lt / den2);
                        if (fabs(rho) > 1.1) { rho = 0; }
                        *out = static_cast<float>(rho);
                    }
                }
            }
        }
        wave_lds_sync();  // the next record rewrites the wave's tables
    }
}

// Split templates: frag[row] = the KT taps of each part in turn (hi, then
// lo for FP16; hi, mid, lo for BF16), zero past Lt.  Each part rounds what
// the parts before it left of the FP64 tap (the remainder is exact in FP64).
template <typename MT>
__global__ __launch_bounds__(NT) void td_prep_kernel(const TdPrepJob *__restrict__ jobs, int KT)
{
    constexpr int NP = TdTraits<MT>::parts;
    const TdPrepJob job = jobs[blockIdx.x];
    MT *f = static_cast<MT *>(job.frag);
    for (int k = threadIdx.x; k < KT; k += NT) {
        double rest = k < job.Lt ? job.tmpl[k] : 0.0;
#pragma unroll
        for (int pt = 0; pt < NP; ++pt) {
            const MT part = static_cast<MT>(static_cast<float>(rest));
            f[pt * KT + k] = part;
            rest -= static_cast<double>(static_cast<float>(part));
        }
    }
}

}  // namespace

hipError_t launch_fix_tiles(const TdRow *dRows, FixQueue queue, int blocks, hipStream_t stream)
{
    if (blocks <= 0 || queue.over == nullptr) { return hipSuccess; }
    hipLaunchKernelGGL(fix_tiles_kernel, dim3(blocks), dim3(NT), 0, stream, dRows, queue);
    return hipGetLastError();
}

bool td_supported(int nb) { return nb >= 1 && nb <= kTdMaxTaps; }

int td_taps(int nb) { return nb <= 64 ? 64 : (nb <= 128 ? 128 : 256); }

hipError_t launch_td_prep(int kind, const TdPrepJob *dJobs, int nJobs, int KT, hipStream_t stream)
{
    if (nJobs <= 0) { return hipSuccess; }
    if (kind == kTdFp16) {
        hipLaunchKernelGGL(td_prep_kernel<_Float16>, dim3(nJobs), dim3(NT), 0, stream, dJobs, KT);
    } else {
        hipLaunchKernelGGL(td_prep_kernel<__bf16>, dim3(nJobs), dim3(NT), 0, stream, dJobs, KT);
    }
    return hipGetLastError();
}

hipError_t launch_td(int kind, int KT, const TdItem *dItems, int nItems, const Seg *dSegs, const TdRow *dRows,
                     FixQueue queue, hipStream_t stream)
{
    if (nItems <= 0) { return hipSuccess; }
#define MF_TD_LAUNCH(MT, K) \
    hipLaunchKernelGGL((tdcorr_kernel<MT, K>), dim3(nItems), dim3(NT), 0, stream, dItems, dSegs, dRows, queue)
    if (kind == kTdFp16) {
        switch (KT) {
        case 64: MF_TD_LAUNCH(_Float16, 64); break;
        case 128: MF_TD_LAUNCH(_Float16, 128); break;
        case 256: MF_TD_LAUNCH(_Float16, 256); break;
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (KT) {
        case 64: MF_TD_LAUNCH(__bf16, 64); break;
        case 128: MF_TD_LAUNCH(__bf16, 128); break;
        case 256: MF_TD_LAUNCH(__bf16, 256); break;
        default: return hipErrorInvalidValue;
        }
    }
#undef MF_TD_LAUNCH
    return hipGetLastError();
}

}  // namespace mfk
