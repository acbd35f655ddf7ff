// Device code of the Toeplitz-block contraction on 16-bit MFMA
// (v_mfma_f32_32x32x16_{bf16,f16}, FP32 accumulation), shared by the kernels
// of fir_mfma.hip (BF16x3, FP16) and fir_f16x2.hip: the split of samples and
// taps into 16-bit terms, the LDS layout of both operands, the contraction of
// one staged segment and its epilogue.
//
// Math (lfilter order, y[n] = sum_k b[k] x[n-k]).  Cut each row's output into
// blocks of 32 samples; block p is y[32p .. 32p+31].  With half-steps
// m = -1 .. m_hi (m_hi = ceil((K-1)/16)):
//   A_m[r][c] = b[16m + r - c]            (32 x 16, zero outside [0, K))
//   B_m[c][p] = x[32p - 16m + c]          (16 x 32 block columns)
//   y[32p + r] = sum_m (A_m B_m)[r][p]
// Each (k, output) pair appears exactly once (m = ceil((k-r)/16), c = 16m-k+r).
//
// Operand reuse.  A wave owns TW output tiles of 32 blocks each, interleaved:
// tile t covers blocks P + t + TW*i (i = 0..31, the MFMA column).  Then tile
// t's B operand at half-step m equals tile 0's at half-step m - 2t, so the
// loop runs over q and every iteration reads ONE B fragment D(q) (tile 0 at
// half-step q) and applies it to tile t with A_{q+2t}.  The A fragments live
// in a ring of 2*TW register sets: each is read once and used by TW tiles.
// Per iteration and split term: one A and one B read for TW MFMAs.
//
// A comes from the taps only.  Each workgroup keeps the split taps in LDS as a
// compact reversed table, T[j] = b[C - j]: lane (i, g) of A_m holds the 8
// consecutive entries starting at j0 = C - 16m - i + 8g (one 16-byte read).
// The table is stored twice, the second copy shifted by one entry, so every
// lane's read is 4-byte aligned; the copies sit 128 bytes apart modulo the
// 256-byte bank cycle.  Entries outside the taps are zero.
//
// B comes from x: the workgroup's segment of 4*TW*32 blocks plus 16*m_hi
// samples of history is split once into LDS.  LDS unit u (8 samples, 16 B)
// of a split array sits at byte 16*(u + u/(4*TW)): lanes read units 4*TW
// apart, and this padding spreads 16 such lanes over distinct bank groups.
//
// Precision modes (template S = number of split terms):
//   S = 3 (BF16x3): v = hi + mid + lo, each bf16 (hi = rn(v), mid = rn(v-hi),
//     lo = rn(v-hi-mid); both subtractions are exact), for x and for b.  Six
//     products are kept: hh (own accumulator), hm, mh, mm, hl, lh (a second
//     accumulator); the dropped ml, lm, ll are below 2^-24 relative.
//   S = 2 (F16x2): v scaled by a power of two, v = hi + 2^-11 lo, each fp16
//     (hi = rn(v), lo = rn(2^11 (v - hi)); the subtraction is exact, lo is
//     within one unit of the last place of v).  Three products are kept: hh in
//     two accumulators (one for each half of the filter), hl and lh together
//     in a third at scale 2^11; the dropped ll is below 2^-22 relative.  What
//     the scaled values have to satisfy is said in fir_f16x2.hip.
//   S = 1 (FP16): x and b rounded to fp16, one product.
// Non-finite values: a zero tap of the Toeplitz block still multiplies its
// sample (and a zero sample its tap), so an Inf or NaN spreads to every output
// of the 32-output blocks it enters, and a finite value beyond the bf16/fp16
// range splits into Inf.  The epilogue therefore recomputes every non-finite
// output from the reference loop's terms (direct_output, FP32 fused
// multiply-add): outputs are non-finite exactly where the reference loop's
// are, at the cost of one class check per output when none is.
//
// MFMA 32x32x16 operand layout (lane l = 32*g + i, g = l/32, i = l%32):
//   A: lane holds A[i][8g + e], e = 0..7;  B: lane holds B[8g + e][i];
//   D: lane holds D[8q + 4g + j][i] in acc[4q + j], q, j = 0..3.
#pragma once

#include "direct_tiles.hpp"
#include "fp16_split.hpp"

#include <algorithm>

namespace scir {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
// Four floats at any 4-byte aligned global address: the kernels load rows and
// store outputs with 16-byte accesses whatever the row's offset or pitch (the
// hardware runs in unaligned access mode; an access that crosses a cache line
// costs two requests, far less than four 4-byte accesses).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxLds = 160 * 1024;
// LDS units (8 samples each) per lane loaded together when a segment's history
// is longer than the prefetched part (2*m_hi > 256 units, K > 2049).
constexpr int kRestBatch = 2;

__host__ __device__ inline int mfma_m_hi(int K) { return (K + 14) / 16; }  // ceil((K-1)/16), K >= 1
inline int mfma_steps(int K) { return mfma_m_hi(K) + 2; }

// Byte address of LDS unit u in a split array whose lanes read 4*TW apart.
template <int TW>
__device__ __forceinline__ int unit_addr(int u)
{
    return (u + u / (4 * TW)) * 16;
}
inline size_t unit_bytes(int units, int tw) { return (size_t)(units + units / (4 * tw) + 1) * 16; }

// Tap table: entries T[j] for j in [0, L), with C chosen so that every A read
// of the loop (half-step indices -2*TW+2 .. msteps+2*TW-1) lands inside it.
inline int tab_C(int m_hi, int tw) { return 16 * (m_hi + 2 * tw + 1) + 32; }
inline int tab_L(int m_hi, int tw) { return tab_C(m_hi, tw) + 32 * tw + 32; }
inline int tab_copy_bytes(int m_hi, int tw)
{
    int bytes = (2 * (tab_L(m_hi, tw) + 1) + 15) & ~15;
    while (bytes % 256 != 128) bytes += 16;
    return bytes;
}

__device__ __forceinline__ unsigned short bf16_bits(__bf16 v) { return __builtin_bit_cast(unsigned short, v); }
__device__ __forceinline__ unsigned short f16_bits(_Float16 v) { return __builtin_bit_cast(unsigned short, v); }

// hi, mid, lo bf16 terms of v (v == hi + mid + lo exactly for normal v).
__device__ __forceinline__ void split3(float v, unsigned short &h, unsigned short &m,
                                       unsigned short &l)
{
    __bf16 bh = (__bf16)v;
    float r1 = v - (float)bh;
    __bf16 bm = (__bf16)r1;
    float r2 = r1 - (float)bm;
    __bf16 bl = (__bf16)r2;
    h = bf16_bits(bh);
    m = bf16_bits(bm);
    l = bf16_bits(bl);
}

// The same split for two values at once, as packed words (v0 in the low half,
// v1 in the high half): one v_cvt_pk_bf16_f32 per term for both values, and
// the words come out in the layout the split arrays store.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned int bf16x2_bits(f32x2 v)
{
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2));
}

__device__ __forceinline__ f32x2 bf16x2_widen(unsigned int w)
{
    return f32x2{__builtin_bit_cast(float, w << 16), __builtin_bit_cast(float, w & 0xffff0000u)};
}

__device__ __forceinline__ void split3_pair(float v0, float v1, unsigned int &h,
                                            unsigned int &m, unsigned int &l)
{
    const f32x2 v = {v0, v1};
    h = bf16x2_bits(v);
    const f32x2 r1 = v - bf16x2_widen(h);
    m = bf16x2_bits(r1);
    const f32x2 r2 = r1 - bf16x2_widen(m);
    l = bf16x2_bits(r2);
}

__device__ __forceinline__ unsigned int pack2(unsigned short lo, unsigned short hi)
{
    return (unsigned int)lo | ((unsigned int)hi << 16);
}

// Tiny magnitudes (BF16x3).  The split terms of v (hi ~ v, mid ~ 2^-8 v,
// lo ~ 2^-16 v) are exact bf16 values, and the kept cross products exact FP32
// values, only while they stay in the normal ranges: for samples and taps
// whose nonzero magnitudes are at least 2^-110, with products of at least
// 2^-100.  A segment whose staged samples or taps go below that (subnormal
// and near-subnormal data) is recomputed from the reference loop's terms.
// Magnitudes are tracked by binary exponent (v = m 2^e, m in [0.5, 1); a
// zero, Inf or NaN gives 0, so it never looks tiny): 2^(e-1) <= |v| < 2^e.
__device__ __forceinline__ int min_exponent(int m, float v)
{
    return min(m, __builtin_amdgcn_frexp_expf(v));
}

__device__ __forceinline__ int wave_min(int v)
{
    return wave_reduce(v, [](int a, int b) { return min(a, b); });
}

// Smallest exponents of the samples (e_x) and taps (e_b) against the limits
// above: 2^(e-1) < 2^-110, or 2^(e_x-1) 2^(e_b-1) < 2^-100.
__device__ __forceinline__ bool tiny_magnitudes(int e_x, int e_b)
{
    return e_x <= -110 || e_b <= -110 || e_x + e_b <= -99;
}

// LDS after the tap tables (after the item slots, ragged): the smallest
// sample exponent of the staged segment per wave, then the taps' per wave.
// Each wave writes its own word after a barrier that every lane passes only
// after reading the previous values, so the words need no reset.
constexpr int kMinsBytes = 32;

// Whether the segment just staged has tiny magnitudes (after the barrier
// that follows staging).
__device__ __forceinline__ bool segment_is_tiny(const int *mins)
{
    const int ex = min(min(mins[0], mins[1]), min(mins[2], mins[3]));
    const int eb = min(min(mins[4], mins[5]), min(mins[6], mins[7]));
    return tiny_magnitudes(ex, eb);
}

template <int S>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c)
{
    if (S == 3)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// acc0 += hi(b)*hi(x); acc1 += the five (BF16x3) or two (F16x2) correction
// products, or acc0 += b*x (FP16).
// FIRST0 / FIRST1: the accumulator's first product (the matrix core takes a
// constant zero, so no register is cleared).
template <int S, bool FIRST0 = false, bool FIRST1 = false>
__device__ __forceinline__ void tile_mfma(f32x16 &acc0, f32x16 &acc1, const u32x4 (&a)[S],
                                          const u32x4 (&d)[S])
{
    constexpr f32x16 zero = {};
    acc0 = mfma<S>(a[0], d[0], FIRST0 ? zero : acc0);
    if (S > 1 && FIRST1) acc1 = zero;
    if (S == 2) {
        constexpr int L = S > 1 ? 1 : 0;
        acc1 = mfma<S>(a[0], d[L], acc1);  // hi(b) * lo(x)
        acc1 = mfma<S>(a[L], d[0], acc1);  // lo(b) * hi(x)
    }
    if (S == 3) {
        constexpr int M = S > 1 ? 1 : 0, L = S > 2 ? 2 : 0;
        acc1 = mfma<S>(a[0], d[M], acc1);  // hi(b) * mid(x)
        acc1 = mfma<S>(a[M], d[0], acc1);  // mid(b) * hi(x)
        acc1 = mfma<S>(a[M], d[M], acc1);  // mid(b) * mid(x)
        acc1 = mfma<S>(a[0], d[L], acc1);  // hi(b) * lo(x)
        acc1 = mfma<S>(a[L], d[0], acc1);  // lo(b) * hi(x)
    }
}

// 16 bytes from a 4-byte aligned LDS address.
__device__ __forceinline__ u32x4 lds_read16_a4(const unsigned char *p)
{
    const unsigned int *q = reinterpret_cast<const unsigned int *>(p);
    return u32x4{q[0], q[1], q[2], q[3]};
}

// Workgroup id -> logical segment id so that the workgroups one XCD receives
// (hardware dispatches id b to XCD b % 8) cover a contiguous range of
// segments: neighbouring segments share their input history in that XCD's L2.
__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t nb)
{
    const int64_t xcd = bid & 7, within = bid >> 3;
    const int64_t q = nb >> 3, rem = nb & 7;
    return xcd * q + (xcd < rem ? xcd : rem) + within;
}

// Loop state of one wave: accumulators, A ring, double-buffered B fragment.
//
// F16x2 runs the half-steps as two passes that end at the middle of the
// filter, the first half upwards, the second downwards, each with its own
// hi*hi accumulator.  A rounded sum errs by its running value, and most
// filters have their large taps in the middle: both sums stay small until
// their last steps: relative L2 0.9e-7 on the 512-tap band-pass, against 1.7e-7
// in one pass, for two more iterations (K = 512: 1795 -> 1830 us).
template <int S, int TW>
struct Contraction {
    static constexpr int RS = 2 * TW;  // A ring slots
    static constexpr int CH = S == 2 ? 2 : 1;  // passes
    f32x16 acc0[CH][TW], acc1[TW];
    u32x4 ring[RS][S];
    u32x4 dA[S], dB[S];
    const unsigned char *lds;
    int ubase;      // B unit of iteration 0 in lane 0 (uniform over the wave)
    int dbase[S];   // the lane's byte address of unit 0 of its column
    int abase[S];   // A table byte address of half-step index 0
    int msteps;     // half-steps per tile

    __device__ __forceinline__ void load_a(u32x4 (&a)[S], int sa) const
    {
#pragma unroll
        for (int s = 0; s < S; ++s) a[s] = lds_read16_a4(lds + abase[s] - 32 * sa);
    }
    __device__ __forceinline__ void load_d(u32x4 (&d)[S], int n) const
    {
        // Lane (i, g) reads unit 4*TW*i + g + u with u even and uniform, so
        // the address is the lane's base plus a scalar (padding included).
        const int u = max(ubase - 2 * n, 0);  // past the last iteration: any in-range unit
#pragma unroll
        for (int s = 0; s < S; ++s)
            d[s] = *reinterpret_cast<const u32x4 *>(lds + dbase[s] + unit_addr<TW>(u));
    }

    enum Mode { kPlain, kPredicated, kFirst };

    // Pass P = 0 takes half-step indices 0 .. count-1 upwards, pass 1
    // msteps-1 .. msteps-count downwards; s counts them.  Iteration n (n % RS
    // == KK): step s = n - 2*TW + 2 + 2t of tile t (pass 1: of tile TW-1-t),
    // whose A is in ring slot (KK + 2 + 2t) % RS, with one D.  After t = 0,
    // whose A is then dead, the slot is refilled with step n + 2.  Predicated,
    // a tile whose s is outside [0, count) is skipped; in the first RS
    // iterations (n == KK) s is a constant, and the accumulators' first
    // products start from zero.
    template <int P>
    __device__ __forceinline__ void load_step_a(u32x4 (&a)[S], int s) const
    {
        load_a(a, P ? msteps - 1 - s : s);
    }
    template <int P>
    __device__ __forceinline__ void load_step_d(u32x4 (&d)[S], int n) const
    {
        load_d(d, P ? msteps + 2 * TW - 3 - n : n);
    }

    template <int P, int KK, Mode M, int T>
    __device__ __forceinline__ void tile(int n, int count, const u32x4 (&dcur)[S])
    {
        constexpr int slot = (KK + 2 + 2 * T) % RS, first_s = KK - 2 * TW + 2 + 2 * T;
        constexpr int t = P ? TW - 1 - T : T;
        if constexpr (M == kFirst && first_s < 0) return;
        const int s = M == kFirst ? first_s : n - 2 * TW + 2 + 2 * T;
        // count >= 1: the first step is there.
        if (M == kPlain || (M == kFirst && first_s == 0) || (s >= 0 && s < count))
            tile_mfma<S, M == kFirst && first_s == 0, P == 0 && M == kFirst && first_s == 0>(
                acc0[P][t], acc1[t], ring[slot], dcur);
    }

    template <int P, int KK, Mode M, int T>
    __device__ __forceinline__ void tiles_from(int n, int count, const u32x4 (&dcur)[S])
    {
        if constexpr (T < TW) {
            tile<P, KK, M, T>(n, count, dcur);
            tiles_from<P, KK, M, T + 1>(n, count, dcur);
        }
    }

    template <int P, int KK, Mode M>
    __device__ __forceinline__ void step(int n, int count)
    {
        u32x4(&dcur)[S] = (KK & 1) ? dB : dA;
        u32x4(&dnxt)[S] = (KK & 1) ? dA : dB;
        load_step_d<P>(dnxt, n + 1);
        __builtin_amdgcn_sched_barrier(0);
        tile<P, KK, M, 0>(n, count, dcur);
        __builtin_amdgcn_sched_barrier(0);
        load_step_a<P>(ring[(KK + 2) % RS], n + 2);
        __builtin_amdgcn_sched_barrier(0);
        tiles_from<P, KK, M, 1>(n, count, dcur);
        __builtin_amdgcn_sched_barrier(0);
    }

    template <int P, int KK>
    __device__ __forceinline__ void tail(int n, int count)
    {
        if constexpr (KK < RS) {
            if (n < count + 2 * TW - 2) {
                step<P, KK, kPredicated>(n, count);
                tail<P, KK + 1>(n + 1, count);
            }
        }
    }

    template <int P, int KK, Mode M>
    __device__ __forceinline__ void body(int n0, int count)
    {
        if constexpr (KK < RS) {
            step<P, KK, M>(n0 + KK, count);
            body<P, KK + 1, M>(n0, count);
        }
    }

    template <int P>
    __device__ __forceinline__ void pass(int count)
    {
        // The ring at iteration 0 holds steps -2TW+2 .. 1 in slot (index mod
        // RS); steps outside the filter read zero table entries.
#pragma unroll
        for (int k = 0; k < RS; ++k) {
            const int s = -2 * TW + 2 + k;
            load_step_a<P>(ring[(k + 2) % RS], s);  // (s mod RS) == (k + 2) mod RS
        }
        load_step_d<P>(dA, 0);
        // The first and last 2TW-2 iterations have tiles outside their steps:
        // the first RS run with the tiles that exist, the last predicated; the
        // rest as unrolled RS-iteration bodies with no branches.
        body<P, 0, kFirst>(0, count);
        int n0 = RS;
        for (; n0 + RS <= count; n0 += RS) {
            if (S == 3 && 2 * n0 >= count) __builtin_amdgcn_s_setprio(1);
            body<P, 0, kPlain>(n0, count);
        }
        // At most RS - 1 + (2TW - 2) < 2*RS iterations remain.
        tail<P, 0>(n0, count);
        tail<P, 0>(n0 + RS, count);
    }

    // Output element e of tile t (F16x2: still at the operands' scale).
    __device__ __forceinline__ float output(int t, int e) const
    {
        if (S == 1) return acc0[0][t][e];
        if (S == 2)
            return acc0[0][t][e] + __builtin_fmaf(acc1[t][e], kLoUnscale, acc0[CH - 1][t][e]);
        return acc0[0][t][e] + acc1[t][e];
    }

    __device__ __forceinline__ void run()
    {
        const int half = CH == 2 ? msteps / 2 : msteps;  // msteps >= 2
        // Of the two waves on a SIMD, the one in the second half of its
        // half-steps goes first, up to its next contraction.  Equal shares
        // keep the two in step, and staging and stores of both then meet
        // (F16x2, K = 512: 1780 -> 1733 us, 1023: 374 -> 355; BF16x3 with its
        // row index stepped, K = 512: 2655 -> 2540).
        if constexpr (S > 1) __builtin_amdgcn_s_setprio(0);
        pass<0>(half);
        if constexpr (CH == 2) {
            __builtin_amdgcn_s_setprio(1);
            pass<1>(msteps - half);
        }
    }
};

// Samples of LDS unit u: 8 samples from xb + 8u of the row (logical order),
// zero outside [0, N) and for u >= units.  With REV logical sample i is
// physical sample N-1-i, and r holds the unit in physical order (slot p =
// logical sample g0 + 7 - p), which unit_sample reads back to front.  Every
// load lands in its slot of r with no register move after it: a move (or a
// select) would wait for the load, and the prefetch of the next segment must
// stay in flight through the contraction.
template <bool REV>
__device__ __forceinline__ void load_unit(const float *__restrict__ xrow, int64_t N, int64_t xb,
                                          int u, int units, f32x4 (&r)[2])
{
    const int64_t g0 = xb + 8 * (int64_t)u;
    if (u >= units) {
        r[0] = r[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    } else if (g0 >= 0 && g0 + 7 < N) {
        const float *p = REV ? xrow + (N - 8 - g0) : xrow + g0;
        r[0] = __builtin_nontemporal_load(reinterpret_cast<const f32x4u *>(p));
        r[1] = __builtin_nontemporal_load(reinterpret_cast<const f32x4u *>(p + 4));
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t i = g0 + e;
            const int slot = REV ? 7 - e : e;
            r[slot >> 2][slot & 3] = 0.0f;
            if (i >= 0 && i < N) r[slot >> 2][slot & 3] = xrow[REV ? N - 1 - i : i];
        }
    }
}

// Logical sample e (0..7) of a unit loaded by load_unit<REV>.
template <bool REV>
__device__ __forceinline__ float unit_sample(const f32x4 (&r)[2], int e)
{
    const int slot = REV ? 7 - e : e;
    return r[slot >> 2][slot & 3];
}

// Split the 8 samples of unit u into the S split arrays of the LDS.
template <int S, int TW, bool REV>
__device__ __forceinline__ void store_unit(unsigned char *lds, int split_stride, int u,
                                           const f32x4 (&r)[2], int &min_e)
{
    if (S == 3) {
        // Smallest binary exponent of the unit's samples: one instruction per
        // sample and a three-input minimum per two.
#pragma unroll
        for (int e = 0; e < 8; e += 2)
            min_e = min(min_e, min(__builtin_amdgcn_frexp_expf(r[e >> 2][e & 3]),
                                   __builtin_amdgcn_frexp_expf(r[e >> 2][(e & 3) + 1])));
        // Pairs in the order the loads left them (slots 2p, 2p + 1).  Back to
        // front, slot pair p holds logical samples 7 - 2p and 6 - 2p, so word
        // 3 - p takes it with its halves swapped.  (Pairs formed from reversed
        // slots made the compiler keep the prefetch registers in scratch.)
        unsigned int w[3][4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            unsigned int h, m, l;
            split3_pair(r[p >> 1][2 * (p & 1)], r[p >> 1][2 * (p & 1) + 1], h, m, l);
            const int q = REV ? 3 - p : p;
            w[0][q] = REV ? __builtin_amdgcn_alignbit(h, h, 16) : h;
            w[1][q] = REV ? __builtin_amdgcn_alignbit(m, m, 16) : m;
            w[2][q] = REV ? __builtin_amdgcn_alignbit(l, l, 16) : l;
        }
#pragma unroll
        for (int s = 0; s < 3; ++s)
            *reinterpret_cast<u32x4 *>(lds + s * split_stride + unit_addr<TW>(u)) =
                u32x4{w[s][0], w[s][1], w[s][2], w[s][3]};
    } else {
        unsigned short t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = f16_bits((_Float16)unit_sample<REV>(r, e));
#pragma unroll
        for (int s = 0; s < S; ++s) {
            u32x4 w = {pack2(t[0], t[1]), pack2(t[2], t[3]), pack2(t[4], t[5]), pack2(t[6], t[7])};
            *reinterpret_cast<u32x4 *>(lds + s * split_stride + unit_addr<TW>(u)) = w;
        }
    }
}

// Tap tables for taps b[0, K) (lfilter order): T_s[j] = split_s(b[C - j]),
// j in [0, L), in two copies one entry apart (copy c holds T_s[pos - c] at
// entry pos, pos in [0, L]), so every lane's 16-byte A read starts 4-byte
// aligned in one of them.  Zero outside the taps.  Each tap is loaded once for
// both copies, four loads in flight per thread before any is used.
template <int S, int TW>
__device__ __forceinline__ void build_tap_table(unsigned char *lds, int tab_offset,
                                                int copy_bytes, const float *__restrict__ b,
                                                int K, int m_hi, int &min_b,
                                                const SplitScale &scale = {})
{
    const int C = 16 * (m_hi + 2 * TW + 1) + 32, L = C + 32 * TW + 32;
    constexpr int R = 4;
    // Entry j in [-1, L]: copy 0 at pos j (j >= 0), copy 1 at pos j + 1 (j < L).
    for (int base = -1; base <= L; base += R * kThreads) {
        float v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int jj = base + (int)threadIdx.x + r * kThreads, k = C - jj;
            v[r] = (jj >= 0 && jj < L && k >= 0 && k < K) ? b[k] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int jj = base + (int)threadIdx.x + r * kThreads;
            if (jj > L) break;
            if (S == 3) min_b = min_exponent(min_b, v[r]);
            unsigned short t[3];
            if (S == 3) {
                split3(v[r], t[0], t[1], t[2]);
            } else if (S == 2) {
                const _Float16 hi = (_Float16)(v[r] * scale.to);
                t[0] = f16_bits(hi);
                t[1] = f16_bits((_Float16)(__builtin_fmaf((float)hi, -scale.from, v[r]) *
                                           scale.to_lo));
            } else {
                t[0] = f16_bits((_Float16)v[r]);
            }
#pragma unroll
            for (int s2 = 0; s2 < S; ++s2) {
                unsigned char *tab = lds + tab_offset + 2 * s2 * copy_bytes;
                if (jj >= 0) *reinterpret_cast<unsigned short *>(tab + 2 * jj) = t[s2];
                if (jj < L)
                    *reinterpret_cast<unsigned short *>(tab + copy_bytes + 2 * (jj + 1)) = t[s2];
            }
        }
    }
    // Every tap load above is consumed, but the compiler cannot tell after the
    // early exit; without this vmcnt(0) it would carry them as pending into
    // the segment loop and wait for each segment's prefetch before the
    // contraction.  (The first segment's samples, loaded before the table,
    // are staged right after this anyway.)
    __builtin_amdgcn_s_waitcnt(0x0f70);
}

// Stage LDS units 0 .. units-1 of a segment (unit 0 = sample xb of the row):
// the first PF units of each lane come from `raw` (loaded ahead), the rest
// are loaded here.
template <int S, int TW, int PF, bool REV>
__device__ __forceinline__ void stage_segment(unsigned char *lds, int split_stride,
                                              const f32x4 (&raw)[PF][2],
                                              const float *__restrict__ xrow, int64_t N,
                                              int64_t xb, int units, int tid, int &min_e)
{
#pragma unroll
    for (int j = 0; j < PF; ++j) {
        const int u = tid + j * kThreads;
        if (u < units) store_unit<S, TW, REV>(lds, split_stride, u, raw[j], min_e);
    }
    if (units <= PF * kThreads) return;  // K <= 2049
    for (int u0 = tid + PF * kThreads; u0 < units; u0 += kRestBatch * kThreads) {
        f32x4 rest[kRestBatch][2];
#pragma unroll
        for (int j = 0; j < kRestBatch; ++j)
            load_unit<REV>(xrow, N, xb, u0 + j * kThreads, units, rest[j]);
#pragma unroll
        for (int j = 0; j < kRestBatch; ++j) {
            const int u = u0 + j * kThreads;
            if (u >= units) break;
            store_unit<S, TW, REV>(lds, split_stride, u, rest[j], min_e);
        }
    }
    // Every load above has been consumed (a unit past `units` is zeros, not
    // loaded), but the compiler cannot tell, and would wait for the next
    // segment's prefetch before the contraction instead: vmcnt(0) here.
    __builtin_amdgcn_s_waitcnt(0x0f70);
}

// Contraction of one staged segment by wave `wave`; lane (i, g) = (lane % 32,
// lane / 32).  The caller's barrier has made the staged units and the tap
// tables visible.
template <int S, int TW>
__device__ __forceinline__ void contract_segment(Contraction<S, TW> &ct, const unsigned char *lds,
                                                 int split_stride, int tab_offset,
                                                 int copy_bytes, int msteps, int m_hi, int wave,
                                                 int i, int g)
{
    const int C = 16 * (m_hi + 2 * TW + 1) + 32;
    ct.lds = lds;
    ct.msteps = msteps;
    // D(n) = tile 0's B at half-step q = n - 2TW + 1: unit
    // 4*(wave offset + TW*i) + 2*(m_hi - q) + g.
    ct.ubase = 128 * TW * __builtin_amdgcn_readfirstlane(wave) + 2 * (m_hi + 2 * TW - 1);
#pragma unroll
    for (int s2 = 0; s2 < S; ++s2)
        ct.dbase[s2] = s2 * split_stride + 16 * (4 * TW + 1) * i + 16 * g;
    {
        // A of half-step index sa (m = sa - 1) starts at entry
        // j0 = C - 16*(sa - 1) - i + 8g, in the copy whose shift c makes j0 + c even.
        const int c = (C - i) & 1;
#pragma unroll
        for (int s2 = 0; s2 < S; ++s2)
            ct.abase[s2] = tab_offset + (2 * s2 + c) * copy_bytes + 2 * (C + 16 - i + 8 * g + c);
    }
    ct.run();
}

// Waits for every load of this wave.  Called after a segment's contraction,
// during which the next segment's samples arrived, and before its stores: the
// samples are then known to be there, and staging them does not wait for the
// stores (loads and stores share one counter), which drain under the next
// contraction.
__device__ __forceinline__ void wait_for_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// What F16x2 adds to a segment's epilogue.
struct SplitOutputs {
    int out_exp = 0;      // the operands' scale, taken back
    float doubt = 0.0f;   // smaller outputs may hang on taps the split has lost
    int m_hi = 0;
};

// Whether the 32 outputs of the workgroup's block `p` see zeros only: their
// staged samples (units from 4p on: the history, then the block).  Nonzero
// samples have a nonzero high term (fir_f16x2.hip's range).
template <int TW>
__device__ __forceinline__ bool silent_block(const unsigned char *lds, int p, int m_hi)
{
    const int end = 4 * p + 2 * m_hi + 4;
#pragma unroll 1
    for (int u = 4 * p; u < end; u += 8) {
        unsigned int any = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // past the end: the last unit again
            const u32x4 w =
                *reinterpret_cast<const u32x4 *>(lds + unit_addr<TW>(min(u + k, end - 1)));
            any |= w.x | w.y | w.z | w.w;
        }
        if (any & 0x7fff7fffu) return false;
    }
    return true;
}

// Epilogue: tile t, lane (i, g) holds block P0 + wave*32*TW + t + TW*i,
// samples 8q + 4g + j; outputs past N are dropped.  A non-finite output, and
// every output of a segment with tiny magnitudes, is recomputed from the
// reference loop's terms (x row xrow, taps b[0, K)).  So is a doubtful one
// (F16x2) among the row's first 16; returns whether the lane has another that
// is not an exact zero of a silent block.
template <int S, int TW, bool REV>
__device__ __forceinline__ bool store_segment(const Contraction<S, TW> &ct,
                                              float *__restrict__ yrow, int64_t N, int64_t P0,
                                              int wave, int i, int g,
                                              const float *__restrict__ xrow,
                                              const float *__restrict__ b, int K, bool tiny,
                                              const SplitOutputs &so = {})
{
    auto output = [&](int t, int e) {
        const float v = ct.output(t, e);
        return S == 2 ? __builtin_ldexpf(v, so.out_exp) : v;
    };
    // Half an instruction per output notes a non-finite one, and half a
    // doubtful one; only such (or a tiny segment) runs a second pass.
    float largest = 0.0f;  // NaN once there is one
    float least[TW], least_head = __builtin_inff();  // a tile's; its first 8 samples of t = 0
    auto note = [&](int t, int q, const f32x4 &v) {
        largest = maximum3(maximum3(largest, v.x, v.y), v.z, v.w);
        if (S != 2) return;
        float &l = t == 0 && q < 2 ? least_head : least[t];
        l = minimum3(minimum3(l, v.x, v.y), v.z, v.w);
    };
    const bool whole = 32 * (P0 + (int64_t)(wave + 1) * 32 * TW) <= N;  // wave-uniform
#pragma unroll
    for (int t = 0; t < TW; ++t) least[t] = __builtin_inff();
    if (whole) {
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            const int64_t n0 = 32 * (P0 + wave * 32 * TW + t + TW * i) + 4 * g;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = output(t, 4 * q + j);
                note(t, q, v);
                const int64_t n = n0 + 8 * q;
                if (!REV)
                    *reinterpret_cast<f32x4u *>(yrow + n) = v;
                else
                    *reinterpret_cast<f32x4u *>(yrow + (N - 4 - n)) = f32x4{v.w, v.z, v.y, v.x};
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            const int64_t n0 = 32 * (P0 + wave * 32 * TW + t + TW * i) + 4 * g;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t n = n0 + 8 * q;
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = output(t, 4 * q + j);
                if (n + 3 < N) {
                    note(t, q, v);
                    if (!REV)
                        *reinterpret_cast<f32x4u *>(yrow + n) = v;
                    else
                        *reinterpret_cast<f32x4u *>(yrow + (N - 4 - n)) =
                            f32x4{v.w, v.z, v.y, v.x};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (n + j < N) {
                            note(t, q, f32x4{v[j], v[j], v[j], v[j]});
                            yrow[REV ? N - 1 - (n + j) : n + j] = v[j];
                        }
                }
            }
        }
    }
    if (tiny || !__builtin_isfinite(largest)) {
        // Over the stored values, in rolled loops: indexing the accumulators
        // there would put them in scratch.
#pragma unroll 1
        for (int t = 0; t < TW; ++t) {
            const int64_t n0 = 32 * (P0 + wave * 32 * TW + t + TW * i) + 4 * g;
#pragma unroll 1
            for (int e = 0; e < 16; ++e) {
                const int64_t n = n0 + 8 * (e >> 2) + (e & 3);
                if (n >= N) break;
                // The thread's own store above, read back.
                float &y = yrow[REV ? N - 1 - n : n];
                if (tiny || !__builtin_isfinite(y))
                    y = direct_output<false>(xrow, N, REV, b, K, n);
            }
        }
    }
    bool more = false;
    if (S == 2 && so.doubt > 0.0f) {
        const bool head = P0 == 0 && wave == 0 && i == 0;
        if (head && least_head < so.doubt) {
            unsigned int which = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                which |= __builtin_fabsf(output(0, e)) < so.doubt ? 1u << e : 0u;
#pragma unroll 1
            for (; which; which &= which - 1) {
                const int e = __builtin_ctz(which);
                const int64_t n = 8 * (e >> 2) + 4 * g + (e & 3);
                if (n < N)
                    yrow[REV ? N - 1 - n : n] = direct_output<false>(xrow, N, REV, b, K, n);
            }
        }
        if (!head) least[0] = fminf(least[0], least_head);
#pragma unroll
        for (int t = 0; t < TW; ++t)
            if (least[t] < so.doubt)
                more |= !silent_block<TW>(ct.lds, wave * 32 * TW + t + TW * i, so.m_hi);
    }
    return more;
}

}  // namespace
}  // namespace scir
