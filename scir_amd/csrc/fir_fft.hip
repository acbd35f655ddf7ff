// FP32 FFT overlap-save FIR for long filters (SCIR_HIP_PREC_FFT32).
//
// The direct and Toeplitz-MFMA kernels cost O(K) per output; a segment of
// NF samples convolved through the FFT costs O(log NF) per output.  Each
// workgroup filters two segments of NF - K + 1 outputs at once: their inputs
// (the K - 1 samples before each plus the segment) are the real and
// imaginary parts of one complex NF-point signal z; since the filter is
// real, IFFT(FFT(z) * H) carries the first segment's circular convolution in
// its real part and the second's in its imaginary part, and entries K-1 ..
// NF-1 of a circular convolution are the linear convolution's outputs.
// H = FFT(b zero-padded to NF) / NF comes from fir_fft_spectrum_kernel,
// launched first on the same stream.  Filters beyond one block of 8192 taps
// run two blocks a pass in fir_fft_pair_kernel, which keeps the spectrum of
// the segment before for the second block.
//
// The transforms run in LDS: radix-16/32 Stockham passes (natural order in
// and out), each thread loading R points with stride NF/R, multiplying by
// the pass twiddles, taking an R-point DFT in registers (radix-2 stages
// with compile-time twiddles) and storing with stride NS.  LDS indices are
// padded by one complex every 32 (i + i/32), which keeps every pass's loads
// and stores free of bank conflicts.  Pass twiddles are products of two
// small tables (64 fine and NF/64 coarse angles) computed on the host in
// double and rounded once.
//
// Error: the FFT's rounding is normwise, about log2(NF) * 2^-24 * |x|_2 |b|_1
// per segment, not relative to each output; the direct and MFMA kernels keep
// the elementwise (K+1) 2^-24 sum|b||x| bound.
//
// Non-finite values: an Inf or NaN anywhere in a segment's window (or an
// overflow inside the transform) makes every output of the segment NaN.  The
// epilogue recomputes each non-finite output from the reference loop's terms
// (direct_output with the whole filter), so outputs are non-finite exactly
// where the reference loop's are.  With a partitioned filter the check is
// made by the block that writes the output last.
#include "direct_tiles.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace scir {
namespace {

// ---- compile-time trigonometry for the in-register DFTs ----------------------
constexpr double kPi = 3.14159265358979323846264338327950288;

constexpr double ct_sin_taylor(double x)
{
    double term = x, sum = x;
    for (int n = 1; n < 30; ++n) {
        term *= -x * x / ((2.0 * n) * (2.0 * n + 1.0));
        sum += term;
    }
    return sum;
}
// cos / sin of 2*pi*m/R
constexpr double ct_cos_frac(int m, int R)
{
    double a = 2.0 * kPi * (double)m / (double)R;
    if (a > kPi) a -= 2.0 * kPi;
    return ct_sin_taylor(a + kPi / 2.0 > kPi ? a + kPi / 2.0 - 2.0 * kPi : a + kPi / 2.0);
}
constexpr double ct_sin_frac(int m, int R)
{
    double a = 2.0 * kPi * (double)m / (double)R;
    if (a > kPi) a -= 2.0 * kPi;
    return ct_sin_taylor(a);
}

template <int R>
struct SmallTw {
    float c[R], s[R];
    constexpr SmallTw() : c(), s()
    {
        for (int m = 0; m < R; ++m) {
            c[m] = (float)ct_cos_frac(m, R);
            s[m] = (float)ct_sin_frac(m, R);
        }
    }
};

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// v <- DFT_R(v) (forward: exp(-2 pi i f n / R); INV: exp(+...)), natural
// order in and out.  Radix-2 decimation in frequency, then the bit-reversal
// permutation (a renaming of registers).
template <int R, bool INV>
__device__ __forceinline__ void dft(float2 (&v)[R])
{
    constexpr SmallTw<R> tw{};
#pragma unroll
    for (int len = R; len >= 2; len >>= 1) {
        const int half = len / 2;
#pragma unroll
        for (int s0 = 0; s0 < R; s0 += len) {
#pragma unroll
            for (int j = 0; j < half; ++j) {
                const float2 a = v[s0 + j], b = v[s0 + j + half];
                v[s0 + j] = cadd(a, b);
                const float2 t = csub(a, b);
                const int m = j * (R / len);  // W_len^j = W_R^m
                if (m == 0) {
                    v[s0 + j + half] = t;
                } else if (4 * m == R) {  // -i (forward) or +i (inverse)
                    v[s0 + j + half] = INV ? make_float2(-t.y, t.x) : make_float2(t.y, -t.x);
                } else {
                    const float2 w = make_float2(tw.c[m], INV ? tw.s[m] : -tw.s[m]);
                    v[s0 + j + half] = cmul(t, w);
                }
            }
        }
    }
    float2 o[R];
#pragma unroll
    for (int f = 0; f < R; ++f) {
        int r = 0;
#pragma unroll
        for (int b = 1, q = f; b < R; b <<= 1, q >>= 1) r = (r << 1) | (q & 1);
        o[f] = v[r];
    }
#pragma unroll
    for (int f = 0; f < R; ++f) v[f] = o[f];
}

__device__ __forceinline__ int pad(int i) { return i + (i >> 5); }

// pad(base + r * NS) - pad(base) for the store pattern of a pass with radix R
// after NS points (base = (j / NS) * NS * R + j % NS): a compile-time offset,
// so the LDS instructions carry it and no per-point address arithmetic is
// left.  NS a multiple of 32: r * NS adds r * NS / 32 pads.  NS == 16 (R
// even): base % 32 < 16, so 16r adds r / 2 pads.  NS == 1, R == 16: base is
// 16j and r < 16 never crosses a 32-point line.
template <int NS, int R>
__device__ __forceinline__ constexpr int store_off(int r)
{
    static_assert(NS % 32 == 0 || (NS == 16 && R % 2 == 0) || (NS == 1 && R == 16),
                  "pass shape without a constant store offset");
    return NS % 32 == 0 ? r * (NS + NS / 32) : NS == 16 ? 16 * r + (r >> 1) : r;
}

// Twiddle tables (cos, sin of positive angles; the forward transform uses
// the conjugates), in this order:
//   tq[i], i < 64:        2*pi*i/NF        (fine)
//   tq[64 + a], a < NF/64: 2*pi*64a/NF      (coarse; fine * coarse gives any
//                                            angle 2*pi*m/NF within ~1.5 ulp)
//   tq[64 + NF/64 + m]:   2*pi*m/(R0*R1)   (the second pass's angles, direct)
//   then, of four passes, 2*pi*m/(R0*R1*R2) (the third pass's)
constexpr int kFine = 64;
template <int NF>
constexpr int tw_fine_coarse() { return kFine + NF / kFine; }

template <int NF, bool INV>
__device__ __forceinline__ float2 twiddle(const float2 *tq, int m)
{
    const float2 p = cmul(tq[m & (kFine - 1)], tq[kFine + m / kFine]);
    return make_float2(p.x, INV ? p.y : -p.y);
}

// One Stockham pass: radix R, NS = product of the earlier radices.
// MULH multiplies the loaded points by the spectrum H first (the pointwise
// product, fused into the inverse transform's first pass).
template <int NF, int T, int R, int NS, bool INV, bool MULH, bool DIRECT = false>
__device__ __forceinline__ void fft_pass(float2 *d, const float2 *tq,
                                         const float2 *__restrict__ H, int tid)
{
    constexpr int B = NF / R;
    constexpr int PER = (B + T - 1) / T;
    static_assert(B % 32 == 0, "loads use pad(j + r*B) == pad(j) + r*(B + B/32)");
    float2 v[PER][R];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int j = tid + p * T;
        if (B % T == 0 || j < B) {
            const int jp = pad(j);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                v[p][r] = d[jp + r * (B + B / 32)];
                if (MULH) {
                    // H[j + r*B] through a buffer resource: the per-point offset
                    // r*B*8 is a scalar constant, so no 64-bit address arithmetic
                    const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(
                        const_cast<float2 *>(H), 0, NF * (int)sizeof(float2), 0x00020000);
                    const float2 h = __builtin_bit_cast(
                        float2, __builtin_amdgcn_raw_buffer_load_b64(hr, 8 * j, 8 * r * B, 0));
                    v[p][r] = cmul(v[p][r], h);
                }
            }
            if (NS > 1) {
                const int k = j % NS;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    float2 w;
                    if (DIRECT) {  // tq points at this pass's table of NS*R angles
                        const float2 t = tq[k * r];
                        w = make_float2(t.x, INV ? t.y : -t.y);
                    } else {
                        w = twiddle<NF, INV>(tq, k * r * (NF / (NS * R)));
                    }
                    v[p][r] = cmul(v[p][r], w);
                }
            }
            dft<R, INV>(v[p]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int j = tid + p * T;
        if (B % T == 0 || j < B) {
            const int k = j % NS;
            const int bp = pad((j / NS) * NS * R + k);
#pragma unroll
            for (int r = 0; r < R; ++r) d[bp + store_off<NS, R>(r)] = v[p][r];
        }
    }
    __syncthreads();
}

template <int LOGN> struct Plan;
template <> struct Plan<12> { static constexpr int T = 256, R0 = 16, R1 = 16, R2 = 16, R3 = 1; };
template <> struct Plan<13> { static constexpr int T = 256, R0 = 16, R1 = 16, R2 = 32, R3 = 1; };
// One workgroup fills a CU's LDS: 16 waves hide more of each other's LDS and
// memory waits than 8 (512 threads, radices 16, 32, 32), for one more pass:
// [256, 262144], K = 8192: 621 -> 505 us, K = 4096: 357 -> 328.
template <> struct Plan<14> { static constexpr int T = 1024, R0 = 16, R1 = 16, R2 = 8, R3 = 8; };

// The passes after the first.  Twiddles: direct tables for the second and, of
// four passes, the third; the last multiplies the fine and the coarse table's.
template <int LOGN, bool INV>
__device__ __forceinline__ void fft_rest(float2 *d, const float2 *tq, int tid)
{
    using P = Plan<LOGN>;
    constexpr int NF = 1 << LOGN, R01 = P::R0 * P::R1;
    // Opaque: the passes of a forward and an inverse transform form the same
    // addresses and twiddle indices, which would be kept from one to the other
    // (the four-pass plan has 128 registers a lane).
    if (P::R3 > 1) asm volatile("" : "+v"(tid));
    const float2 *direct = tq + tw_fine_coarse<NF>();
    fft_pass<NF, P::T, P::R1, P::R0, INV, false, true>(d, direct, nullptr, tid);
    if constexpr (P::R3 > 1) {
        fft_pass<NF, P::T, P::R2, R01, INV, false, true>(d, direct + R01, nullptr, tid);
        fft_pass<NF, P::T, P::R3, R01 * P::R2, INV, false>(d, tq, nullptr, tid);
    } else {
        fft_pass<NF, P::T, P::R2, R01, INV, false>(d, tq, nullptr, tid);
    }
}

template <int LOGN, bool INV, bool MULH>
__device__ __forceinline__ void fft(float2 *d, const float2 *tq, const float2 *__restrict__ H,
                                    int tid)
{
    using P = Plan<LOGN>;
    fft_pass<1 << LOGN, P::T, P::R0, 1, INV, MULH>(d, tq, H, tid);
    fft_rest<LOGN, INV>(d, tq, tid);
}

template <int LOGN>
constexpr int tw_entries()
{
    using P = Plan<LOGN>;
    return tw_fine_coarse<1 << LOGN>() + P::R0 * P::R1 + (P::R3 > 1 ? P::R0 * P::R1 * P::R2 : 0);
}

template <int LOGN>
constexpr size_t lds_bytes()
{
    constexpr int NF = 1 << LOGN;
    return (size_t)(NF + NF / 32 + tw_entries<LOGN>()) * sizeof(float2);
}

// Taps per block of the FFT path: the largest transform (2^14) keeps at
// least half of each segment as outputs.  Longer filters are cut into blocks
// of kFftBlockTaps taps (uniformly partitioned overlap-save): block j, taps
// b[jP, jP + P), filters the input delayed by jP samples.
constexpr int kFftBlockTaps = 8192;

// H[i] = FFT(b zero-padded)[i] / NF, one workgroup for each block of taps.
template <int LOGN>
__global__ __launch_bounds__(Plan<LOGN>::T) void fir_fft_spectrum_kernel(
    const float *__restrict__ b, int K, const float2 *__restrict__ tq_g, float2 *__restrict__ H)
{
    constexpr int NF = 1 << LOGN, T = Plan<LOGN>::T;
    b += (int)blockIdx.x * kFftBlockTaps;
    K = min(K - (int)blockIdx.x * kFftBlockTaps, kFftBlockTaps);
    H += (int64_t)blockIdx.x * NF;
    extern __shared__ float2 lds_f2[];
    float2 *d = lds_f2;
    float2 *tq = lds_f2 + NF + NF / 32;
    const int tid = threadIdx.x;
    for (int i = tid; i < tw_entries<LOGN>(); i += T) tq[i] = tq_g[i];
    for (int i = tid; i < NF; i += T) d[pad(i)] = make_float2(i < K ? b[i] : 0.0f, 0.0f);
    __syncthreads();
    fft<LOGN, false, false>(d, tq, nullptr, tid);
    const float inv = 1.0f / (float)NF;  // exact: NF is a power of two
    for (int i = tid; i < NF; i += T) {
        const float2 v = d[pad(i)];
        H[i] = make_float2(v.x * inv, v.y * inv);
    }
}

// Segment s of the (row, segment) list: row s / spr, outputs [o, o + V),
// V = NF - K + 1, o = (s % spr) * V.  REV reads and writes every row back to
// front (the anti-causal correlation of the dL/dx adjoint).  With `accumulate`
// the outputs are added to y instead of stored (the later tap blocks of a
// partitioned filter).  The block holds taps bfull[j0, j0 + K) of a filter of
// Kfull taps: its output t is output t + j0 of the whole filter, its input t
// is the row's input t, and it writes outputs t < final_len last (the later
// blocks start at t = kFftBlockTaps).
template <int LOGN, bool REV>
__global__ __launch_bounds__(Plan<LOGN>::T) void fir_fft_kernel(
    const float *__restrict__ x, int64_t ldx, float *__restrict__ y, int64_t ldy, int64_t N,
    int K, const float2 *__restrict__ H, const float2 *__restrict__ tq_g, int64_t spr,
    int64_t nseg, int accumulate, const float *__restrict__ bfull, int Kfull, int64_t j0,
    int64_t final_len)
{
    constexpr int NF = 1 << LOGN, T = Plan<LOGN>::T;
    extern __shared__ float2 lds_f2[];
    float2 *d = lds_f2;
    float2 *tq = lds_f2 + NF + NF / 32;
    const int tid = threadIdx.x;
    const int V = NF - K + 1;
    const int64_t s0 = 2 * (int64_t)blockIdx.x, s1 = s0 + 1;
    const bool has1 = s1 < nseg;
    const int64_t ra = s0 / spr, oa = (s0 - ra * spr) * V;
    const int64_t rb = has1 ? s1 / spr : ra, ob = has1 ? (s1 - rb * spr) * V : 0;
    const float *xa = x + ra * ldx, *xb = x + rb * ldx;
    for (int i = tid; i < tw_entries<LOGN>(); i += T) tq[i] = tq_g[i];
    const int64_t wa = oa - (K - 1), wb = ob - (K - 1);  // first input of each window
    if (has1 && wa >= 0 && wa + NF <= N && wb >= 0 && wb + NF <= N) {
        // both windows inside their rows: no bounds checks
        const float *pa = REV ? xa + (N - 1 - wa) : xa + wa;
        const float *pb = REV ? xb + (N - 1 - wb) : xb + wb;
        // pad(tid + m*T) == pad(tid) + m*(T + T/32): T is a multiple of 32
        static_assert(T % 32 == 0, "constant LDS offsets need T % 32 == 0");
        const int tp = pad(tid);
#pragma unroll 4
        for (int m = 0; m < NF / T; ++m) {
            const int i = tid + m * T;
            d[tp + m * (T + T / 32)] = make_float2(pa[REV ? -i : i], pb[REV ? -i : i]);
        }
    } else {
        for (int i = tid; i < NF; i += T) {
            const int64_t ta = wa + i, tb = wb + i;
            float va = 0.0f, vb = 0.0f;
            if (ta >= 0 && ta < N) va = xa[REV ? N - 1 - ta : ta];
            if (has1 && tb >= 0 && tb < N) vb = xb[REV ? N - 1 - tb : tb];
            d[pad(i)] = make_float2(va, vb);
        }
    }
    __syncthreads();
    fft<LOGN, false, false>(d, tq, nullptr, tid);
    fft<LOGN, true, true>(d, tq, H, tid);
    float *ya = y + ra * ldy, *yb = y + rb * ldy;
    // The rows of the whole filter (for recomputing non-finite outputs): in
    // REV mode the block's rows start j0 samples into the physical row.
    const float *fa = REV ? xa - j0 : xa, *fb = REV ? xb - j0 : xb;
    const int64_t Nf = N + j0;
    auto finish = [&](float v, const float *frow, int64_t t) {
        if (!__builtin_isfinite(v) && t < final_len)
            v = direct_output<false>(frow, Nf, REV, bfull, Kfull, t + j0);
        return v;
    };
    if (has1 && oa + V <= N && ob + V <= N) {
        float *qa = REV ? ya + (N - 1 - oa) : ya + oa;
        float *qb = REV ? yb + (N - 1 - ob) : yb + ob;
        // Outputs are stored as computed; a flag notes whether any came out
        // non-finite (one class test each, no branch in the loop), and only
        // then are the thread's outputs read back and fixed.
        bool bad = false;
        if (accumulate) {
#pragma unroll 4
            for (int v = tid; v < V; v += T) {
                const float2 o = d[pad(K - 1 + v)];
                float &pa = qa[REV ? -v : v], &pb = qb[REV ? -v : v];
                const float a = pa + o.x, b = pb + o.y;
                pa = a;
                pb = b;
                bad |= !__builtin_isfinite(a) | !__builtin_isfinite(b);
            }
        } else {
#pragma unroll 4
            for (int v = tid; v < V; v += T) {
                const float2 o = d[pad(K - 1 + v)];
                qa[REV ? -v : v] = o.x;
                qb[REV ? -v : v] = o.y;
                bad |= !__builtin_isfinite(o.x) | !__builtin_isfinite(o.y);
            }
        }
        if (bad) {
            for (int v = tid; v < V; v += T) {
                float &pa = qa[REV ? -v : v], &pb = qb[REV ? -v : v];
                pa = finish(pa, fa, oa + v);
                pb = finish(pb, fb, ob + v);
            }
        }
    } else {
        for (int v = tid; v < V; v += T) {
            const float2 o = d[pad(K - 1 + v)];
            const int64_t ta = oa + v, tb = ob + v;
            if (ta < N) {
                float &q = ya[REV ? N - 1 - ta : ta];
                q = finish(accumulate ? q + o.x : o.x, fa, ta);
            }
            if (has1 && tb < N) {
                float &q = yb[REV ? N - 1 - tb : tb];
                q = finish(accumulate ? q + o.y : o.y, fb, tb);
            }
        }
    }
}

// Two blocks of taps in one pass: y_s = IFFT(X_s H0 + X_{s-1} H1) with X_s the
// transform of the window [8192 (s-1), 8192 (s+1)) of segment s.  A workgroup
// walks a run of segments of two streams (rows, or runs of one row), which are
// the real and imaginary parts of one signal.  Each thread keeps the 16 points
// of X_{s-1} that it multiplies, so a segment costs one transform each way and
// its outputs are written once; block by block it cost two of each (and a read
// and a write of y): [256, 262144], K = 16384: 1173 -> 446 us.
// One workgroup fits a CU (153 KB of LDS), so the transforms' LDS phases and
// arithmetic alternate; that, not memory, bounds it.
// A run that does not start its row first transforms the window before it.
template <bool REV>
__global__ __launch_bounds__(Plan<14>::T) void fir_fft_pair_kernel(
    const float *__restrict__ x, int64_t ldx, float *__restrict__ y, int64_t ldy, int64_t N,
    const float2 *__restrict__ H, const float2 *__restrict__ tq_g, int64_t spr, int64_t run,
    int64_t runs_per_row, int64_t streams, int accumulate, const float *__restrict__ bfull,
    int Kfull, int64_t j0, int64_t final_len)
{
    using P = Plan<14>;
    constexpr int NF = 1 << 14, T = P::T, SEG = kFftBlockTaps, M = SEG / T;
    constexpr int R0 = P::R0, B0 = NF / R0;  // the inverse transform's first pass
    static_assert(2 * SEG == NF && SEG % T == 0 && B0 == T && T % 32 == 0, "pass shapes");
    extern __shared__ float2 lds_f2[];
    float2 *d = lds_f2;
    float2 *tq = lds_f2 + NF + NF / 32;
    int tid = threadIdx.x;
    for (int i = tid; i < tw_entries<14>(); i += T) tq[i] = tq_g[i];

    struct Stream {
        const float *x;
        float *y;
        int64_t seg0, count;  // first segment, segments
    };
    auto stream = [&](int64_t u) {
        if (u >= streams) return Stream{x, y, 0, 0};
        const int64_t row = u / runs_per_row, s0 = (u - row * runs_per_row) * run;
        return Stream{x + row * ldx, y + row * ldy, s0, min(run, spr - s0)};
    };
    const Stream sa = stream(2 * (int64_t)blockIdx.x), sb = stream(2 * (int64_t)blockIdx.x + 1);
    const int64_t steps = max(sa.count, sb.count);

    auto lane = [&]() { return (unsigned int)(REV ? T - 1 - tid : tid); };
    // The window of segment `seg` of one stream, samples tid + T m; zeros
    // outside the row and past the stream's run.
    auto load = [&](const Stream &st, int64_t seg, bool wanted, float (&v)[2 * M]) {
        const int64_t t0 = (seg - 1) * SEG;
        if (wanted && t0 >= 0 && t0 + NF <= N) {
            // A uniform base and a 32-bit lane offset.
#pragma unroll
            for (int m = 0; m < 2 * M; ++m)
                v[m] = (REV ? st.x + (N - t0 - T * (m + 1)) : st.x + (t0 + T * m))[lane()];
        } else {
#pragma unroll
            for (int m = 0; m < 2 * M; ++m) {
                const int64_t t = t0 + tid + T * m;
                v[m] = 0.0f;
                if (wanted && t >= 0 && t < N) v[m] = st.x[REV ? N - 1 - t : t];
            }
        }
    };
    float wa[2 * M], wb[2 * M];
    auto fill = [&]() {
#pragma unroll
        for (int m = 0; m < 2 * M; ++m)
            d[pad(tid) + m * (T + T / 32)] = make_float2(wa[m], wb[m]);
        __syncthreads();
    };
    float2 prev[R0];  // X_{s-1} at tid + B0 r
#pragma unroll
    for (int r = 0; r < R0; ++r) prev[r] = make_float2(0.0f, 0.0f);
    if (sa.seg0 > 0 || sb.seg0 > 0) {
        load(sa, sa.seg0 - 1, sa.count > 0, wa);
        load(sb, sb.seg0 - 1, sb.count > 0, wb);
        fill();
        fft<14, false, false>(d, tq, nullptr, tid);
#pragma unroll
        for (int r = 0; r < R0; ++r) prev[r] = d[pad(tid) + r * (B0 + B0 / 32)];
        __syncthreads();
    }
    load(sa, sa.seg0, sa.count > 0, wa);
    load(sb, sb.seg0, sb.count > 0, wb);

    // The rows of the whole filter (for recomputing non-finite outputs): in
    // REV mode the block's rows start j0 samples into the physical row.
    const int64_t Nf = N + j0;
    auto finish = [&](const Stream &st, float v, int64_t t) {
        if (!__builtin_isfinite(v) && t < final_len)
            v = direct_output<false>(REV ? st.x - j0 : st.x, Nf, REV, bfull, Kfull, t + j0);
        return v;
    };
    const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float2 *>(H), 0, 2 * NF * (int)sizeof(float2), 0x00020000);
    for (int64_t i = 0; i < steps; ++i) {
        asm volatile("" : "+v"(tid));  // as in fft_rest
        fill();
        fft<14, false, false>(d, tq, nullptr, tid);
        {  // the inverse transform's first pass (fft_pass), with the products
            float2 v[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const float2 X = d[pad(tid) + r * (B0 + B0 / 32)];
                const float2 h0 = __builtin_bit_cast(float2,
                    __builtin_amdgcn_raw_buffer_load_b64(hr, 8 * tid, 8 * r * B0, 0));
                const float2 h1 = __builtin_bit_cast(float2,
                    __builtin_amdgcn_raw_buffer_load_b64(hr, 8 * tid, 8 * (NF + r * B0), 0));
                v[r] = cadd(cmul(X, h0), cmul(prev[r], h1));
                prev[r] = X;
                // Spectra of four points in registers at a time.
                if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            dft<R0, true>(v);
            __syncthreads();
            const int bp = pad(tid * R0);
#pragma unroll
            for (int r = 0; r < R0; ++r) d[bp + store_off<1, R0>(r)] = v[r];
            __syncthreads();
        }
        fft_rest<14, true>(d, tq, tid);
        // The next window loads while the outputs go out (no earlier: the
        // transforms need the registers).
        load(sa, sa.seg0 + i + 1, i + 1 < sa.count, wa);
        load(sb, sb.seg0 + i + 1, i + 1 < sb.count, wb);
        auto store = [&](const Stream &st, bool imag) {
            if (i >= st.count) return;
            const int64_t t0 = (st.seg0 + i) * SEG;
            bool bad = false;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float2 o = d[pad(tid) + (m + M) * (T + T / 32)];
                if (t0 + tid + T * m >= N) break;
                float out = imag ? o.y : o.x;
                float &at = (REV ? st.y + (N - t0 - T * (m + 1)) : st.y + (t0 + T * m))[lane()];
                if (accumulate) out += at;
                at = out;
                bad |= !__builtin_isfinite(out);
            }
            if (bad)
                for (int v = tid; v < SEG && t0 + v < N; v += T) {
                    float &at = st.y[REV ? N - 1 - (t0 + v) : t0 + v];
                    at = finish(st, at, t0 + v);
                }
        };
        store(sa, false);
        store(sb, true);
        __syncthreads();
    }
}

// Twiddle tables, one per size, built on first use per device (kept in the
// device state, freed by scir_hip_shutdown).
int twiddle_table(DeviceState *st, int logn, hipStream_t s, const float2 **out)
{
    const int NF = 1 << logn;
    DeviceBuffer &buf = st->fft_twiddles[logn - 12];
    if (!buf.ptr) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (s != nullptr && hipStreamIsCapturing(s, &cs) == hipSuccess &&
            cs != hipStreamCaptureStatusNone)
            return fail(SCIR_HIP_ERR_CAPTURE,
                        "the FFT twiddle table is built on first use; run once outside capture");
        // Direct tables of Plan<logn>: R0 * R1 angles, and R0 * R1 * R2.
        std::vector<int> direct(1, 256);
        if (logn == 14) direct.push_back(2048);
        std::vector<float2> h;
        h.reserve(kFine + NF / kFine + 2304);
        h.resize(kFine + NF / kFine);
        for (int i = 0; i < kFine; ++i) {
            const double a = 2.0 * kPi * (double)i / (double)NF;
            h[i] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
        for (int i = 0; i < NF / kFine; ++i) {
            const double a = 2.0 * kPi * (double)(i * kFine) / (double)NF;
            h[kFine + i] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
        for (int n : direct)
            for (int m = 0; m < n; ++m) {
                const double a = 2.0 * kPi * (double)m / (double)n;
                h.push_back(make_float2((float)std::cos(a), (float)std::sin(a)));
            }
        void *p = nullptr;
        SCIR_TRY(device_alloc(&p, h.size() * sizeof(float2), "FFT twiddle table"));
        const hipError_t e = hipMemcpy(p, h.data(), h.size() * sizeof(float2),
                                       hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(p);
            return fail(SCIR_HIP_ERR_BACKEND, "FFT twiddle upload failed: %s",
                        hipGetErrorString(e));
        }
        buf.ptr = p;
        buf.bytes = h.size() * sizeof(float2);
    }
    *out = static_cast<const float2 *>(buf.ptr);
    return SCIR_HIP_OK;
}

// Spectra of `blocks` blocks of the K taps at b, on stream s: *H (and *tq, the
// twiddle table) for the filter kernels.
template <int LOGN>
int filter_spectra(const float *b, int K, int blocks, hipStream_t s, DeviceState *st,
                   const float2 **tq, float2 **H)
{
    constexpr int NF = 1 << LOGN;
    constexpr size_t lds = lds_bytes<LOGN>();
    SCIR_TRY(twiddle_table(st, LOGN, s, tq));
    StreamScratch &sc = scratch_for(st, s);
    // The largest size holds two spectra from the start: a filter of more
    // blocks then needs no more scratch than one of fewer.
    SCIR_TRY(ensure_scratch(st, sc.fft_spectrum,
                            (size_t)(LOGN == 14 ? 2 : 1) * NF * sizeof(float2), s));
    *H = static_cast<float2 *>(sc.fft_spectrum.ptr);
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(&fir_fft_spectrum_kernel<LOGN>),
                               (int)lds));
    hipLaunchKernelGGL((fir_fft_spectrum_kernel<LOGN>), dim3((unsigned)blocks),
                       dim3(Plan<LOGN>::T), lds, s, b, K, *tq, *H);
    return check_launch("fir_fft_spectrum_kernel");
}

template <int LOGN>
int launch_fft(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N, float *y,
               int64_t ldy, bool rev, bool accumulate, const float *bfull, int Kfull, int64_t j0,
               int64_t final_len, hipStream_t s, DeviceState *st)
{
    constexpr int NF = 1 << LOGN, T = Plan<LOGN>::T;
    const float2 *tq = nullptr;
    float2 *H = nullptr;
    SCIR_TRY(filter_spectra<LOGN>(b, K, 1, s, st, &tq, &H));
    constexpr size_t lds = lds_bytes<LOGN>();
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(&fir_fft_kernel<LOGN, false>),
                               (int)lds));
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(&fir_fft_kernel<LOGN, true>),
                               (int)lds));
    const int64_t V = NF - K + 1;
    const int64_t spr = (N + V - 1) / V;
    const int64_t nseg = B * spr;
    const int64_t blocks = (nseg + 1) / 2;
    if (blocks > 0x7fffffff) return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "batch too large");
    const int acc = accumulate ? 1 : 0;
    if (rev)
        hipLaunchKernelGGL((fir_fft_kernel<LOGN, true>), dim3((unsigned)blocks), dim3(T), lds, s, x,
                           ldx, y, ldy, N, K, H, tq, spr, nseg, acc, bfull, Kfull, j0, final_len);
    else
        hipLaunchKernelGGL((fir_fft_kernel<LOGN, false>), dim3((unsigned)blocks), dim3(T), lds, s,
                           x, ldx, y, ldy, N, K, H, tq, spr, nseg, acc, bfull, Kfull, j0,
                           final_len);
    return check_launch("fir_fft_kernel");
}

// FFT size for K taps: the smallest of 2^12, 2^13, 2^14 with NF >= 4K
// (outputs per segment >= 3/4 NF), else 2^14.
int fft_log_size(int K)
{
    if (4 * K <= 4096) return 12;
    if (4 * K <= 8192) return 13;
    return 14;
}

int fft_block(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N, float *y,
              int64_t ldy, bool rev, bool accumulate, const float *bfull, int Kfull, int64_t j0,
              int64_t final_len, hipStream_t stream, DeviceState *st)
{
#define SCIR_FFT_BLOCK(L)                                                                      \
    launch_fft<L>(x, ldx, b, K, B, N, y, ldy, rev, accumulate, bfull, Kfull, j0, final_len, \
                  stream, st)
    switch (fft_log_size(K)) {
    case 12: return SCIR_FFT_BLOCK(12);
    case 13: return SCIR_FFT_BLOCK(13);
    default: return SCIR_FFT_BLOCK(14);
    }
#undef SCIR_FFT_BLOCK
}

// Two blocks of taps (K of them at b, more than kFftPairMinTaps) in one pass.
constexpr int kFftPairMinTaps = 7168;

int fft_block_pair(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                   float *y, int64_t ldy, bool rev, bool accumulate, const float *bfull,
                   int Kfull, int64_t j0, int64_t final_len, hipStream_t s, DeviceState *st)
{
    const float2 *tq = nullptr;
    float2 *H = nullptr;
    SCIR_TRY(filter_spectra<14>(b, K, 2, s, st, &tq, &H));
    constexpr size_t lds = lds_bytes<14>();
    const int64_t spr = (N + kFftBlockTaps - 1) / kFftBlockTaps;
    // Runs per row: the fewest rounds of workgroups over the CUs times a run's
    // cost (its segments, and half of one for the window before it).
    const int64_t cus = std::max(1, st->cu_count);
    int64_t runs = 1;
    double best = 1e30;
    for (int64_t c = 1; c <= spr && c <= 4 * cus; ++c) {
        const int64_t len = (spr + c - 1) / c, n = (spr + len - 1) / len;
        const int64_t rounds = ((B * n + 1) / 2 + cus - 1) / cus;
        const double cost = (double)rounds * ((double)len + (n > 1 ? 0.5 : 0.0));
        if (cost < best) {
            best = cost;
            runs = n;
        }
    }
    const int64_t run = (spr + runs - 1) / runs;
    runs = (spr + run - 1) / run;
    const int64_t blocks = (B * runs + 1) / 2;
    if (blocks > 0x7fffffff) return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "batch too large");
    auto *kernel = rev ? &fir_fft_pair_kernel<true> : &fir_fft_pair_kernel<false>;
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(kernel), (int)lds));
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(Plan<14>::T), lds, s, x, ldx, y, ldy,
                       N, H, tq, spr, run, runs, B * runs, accumulate ? 1 : 0, bfull, Kfull, j0,
                       final_len);
    return check_launch("fir_fft_pair_kernel");
}

}  // namespace

int fir_fft_dev(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N, float *y,
                int64_t ldy, bool rev, hipStream_t stream, DeviceState *st)
{
    if (K == 0)  // no taps: zeros, as every path gives
        return fir_direct_dev(x, ldx, b, K, B, N, y, ldy, false, rev, stream, st);
    if (K < 0) return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "negative tap count");
    if (x == y)
        return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "the FFT path does not filter in place");
    if (B == 0 || N == 0) return SCIR_HIP_OK;
    for (int64_t j0 = 0, step; j0 < K && j0 < N; j0 += step) {
        // Two blocks at once, also when the second has no taps but the first
        // leaves fft_block few outputs a segment ([256, 262144], K = 8192: 505
        // us by fft_block, 446 by the pair; they cross at about 7100).
        const bool pair = K - j0 > kFftPairMinTaps && N - j0 > kFftBlockTaps;
        step = pair ? 2 * kFftBlockTaps : kFftBlockTaps;
        const int Kj = (int)std::min<int64_t>(step, K - j0);
        // Forward: y[j0 + i] += sum_k b[j0 + k] x[i - k] for i < N - j0.  Back
        // to front the same sums read x from sample j0 on and write y from 0.
        const float *xs = rev ? x + j0 : x;
        float *ys = rev ? y : y + j0;
        // This pass writes outputs j0 .. j0 + step - 1 last (all the rest when
        // it is the final one).
        const bool last = j0 + step >= K || j0 + step >= N;
        const int64_t final_len = last ? N - j0 : step;
        SCIR_TRY((pair ? fft_block_pair : fft_block)(xs, ldx, b + j0, Kj, B, N - j0, ys, ldy, rev,
                                                     j0 > 0, b, K, j0, final_len, stream, st));
    }
    return SCIR_HIP_OK;
}

}  // namespace scir
