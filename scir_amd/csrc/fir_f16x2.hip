// F32 filters of medium length on the 16-bit matrix cores: the Toeplitz-block
// contraction of toeplitz_mfma.hpp with samples and taps split into two fp16
// terms (F16x2, three products), dense and ragged.
//
// Why two fp16 terms.  The FP32 matrix cores do 157 TFLOP/s and the BF16x3
// split spends six bf16 products a tap; hi + 2^-11 lo in fp16 carries 23 bits
// (FP32 has 24) with three products at the same rate, and LDS holds two split
// arrays instead of three.  Its error against 64 bits is below the FP32
// kernels' at every length it is chosen for (rounded sums dominate theirs):
// relative L2 0.8e-7 against 2.0e-7 of the FP32 matrix cores at K = 129,
// 0.9e-7 / 3.9e-7 at 512, 0.9e-7 / 5.4e-7 of the VALU form at 1023.
//
// Measured, us a call (before: the FP32 matrix cores to K = 513, the VALU
// above; in brackets BF16x3):
//   [4096, 65536]   K = 129   698 -> 515  (600)    255  1274 -> 612  (810)
//   [2048, 262144]  K = 512  5550 -> 1733 (2540)
//   [1024, 65536]   K = 1023 1818 -> 350  (600)   2040  3572 -> 610 (1060)
//   2500 ragged signals, K 15 .. 1023: 4370 -> 1080 (1625)
// At K = 512 the matrix cores are busy 61 % of the cycles at a clock that the
// load pulls down to 1.4 GHz (with one workgroup a CU it runs at 1.9), so the
// bound is power; below K = 200 it is HBM and the phases that do not overlap
// (staging and stores of one wave against the contraction of the other on its
// SIMD).
//
// Range.  fp16 has five exponent bits, so samples and taps are scaled by
// powers of two: the taps by 2^sb, which puts the largest in [2^13, 2^14), the
// samples of each segment (with its history) by 2^sx, chosen the same way.
// With X, B the scaled values, hi and lo are exact to half a unit of fp16's
// subnormal grid (matrix cores keep fp16 subnormals), i.e. |error of X| <=
// max(2^-23 |X|, 2^-36), and the dropped lo * lo is as small.  The bound of
// F32, (K+1) 2^-23 sum |b||x|, therefore holds when
//   * every nonzero |X| >= 2^-T with T = 10 + floor(log2(K + 1)) (its floor of
//     2^-36 is at most (K+1) 2^-26 of its term), and
//   * taps below 2^-14 (the zero crossings of a sinc come out as 1e-17, not
//     as 0), whose errors are at most err = sum min(|B|, 2^-35), do not carry
//     an output alone.  They do not where |Y| >= 2 err max|X| / ((K+1) 2^-25),
//     for |Y| is a lower bound of sum |B||X| (up to the errors, hence the 2):
//     about 1e-9 of full scale.  Of smaller outputs, the row's first 16 (a
//     first tap that is almost zero) are recomputed from the reference loop's
//     terms, those that see zeros only are exact, and a segment with others
//     (impulses in silence) is filtered again by BF16x3.  (Ruling such
//     segments out from the samples' and the taps' magnitudes instead sent
//     every segment with a zero sample to BF16x3: ten zeros in 67 million
//     samples cost 37 of 370 us.)
// A segment outside the first limit (and every segment of a filter of fewer
// than 16 taps, where the bound leaves no room, or of one with an Inf) is
// filtered by the BF16x3 contraction in the same workgroup, half a segment at
// a time.  The choice and the scale depend on the segment's samples and the
// taps alone, so the result does not depend on how segments are grouped.
#include "toeplitz_mfma.hpp"

namespace scir {
namespace {

constexpr int kMinTaps = 16;      // fewer: always BF16x3
constexpr int kMaxTaps = 2049;    // history units fit the prefetched ones (m_hi <= 128)

// Words of LDS the waves exchange: per wave (4) unless said otherwise.
enum Word {
    kSampleMax = 0,    // |x| bits, of the next segment to stage
    kSampleExp = 4,    // smallest exponent of a nonzero sample
    kTapErr = 8,       // bound of the errors of the taps below 2^-14
    kTapMax = 12,      // |b| bits
    kRedo = 16,        // the wave has doubtful outputs
    kMins3 = 20,       // 8 words: the BF16x3 path's exponents
    kWords = 28
};

// LDS: two split arrays of a segment (or three of half a segment), the tap
// tables of either split, the words.
struct F16x2Layout {
    int stride2, stride3, tab_offset, copy2, copy3, words_offset;
};

F16x2Layout f16x2_layout(int K, int tw)
{
    const int m_hi = mfma_m_hi(K);
    F16x2Layout l;
    l.stride2 = (int)unit_bytes(kWaves * tw * 128 + 2 * m_hi, tw);
    l.stride3 = (int)unit_bytes(kWaves * 128 + 2 * m_hi, 1);
    l.tab_offset = std::max(2 * l.stride2, 3 * l.stride3);
    l.copy2 = tab_copy_bytes(m_hi, tw);
    l.copy3 = tab_copy_bytes(m_hi, 1);
    l.words_offset = l.tab_offset + std::max(4 * l.copy2, 6 * l.copy3);
    return l;
}
inline size_t f16x2_lds(const F16x2Layout &l) { return (size_t)l.words_offset + 4 * kWords + 16; }

// Splits the 8 samples of unit u into the two split arrays.
template <int TW, bool REV>
__device__ __forceinline__ void store_unit2(unsigned char *lds, int stride, int u,
                                            const f32x4 (&r)[2], const SplitScale &scale)
{
    unsigned int w[2][4];
#pragma unroll
    for (int p = 0; p < 4; p += 2) {
        unsigned int h[2], l[2];
        split2_quad(r[p >> 1], scale, h, l);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int q = REV ? 3 - p - e : p + e;  // as in store_unit
            w[0][q] = REV ? __builtin_amdgcn_alignbit(h[e], h[e], 16) : h[e];
            w[1][q] = REV ? __builtin_amdgcn_alignbit(l[e], l[e], 16) : l[e];
        }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
        *reinterpret_cast<u32x4 *>(lds + s * stride + unit_addr<TW>(u)) =
            u32x4{w[s][0], w[s][1], w[s][2], w[s][3]};
}

// One workgroup's state: the filter, the scales and what its LDS holds.
template <int TW, bool REV>
struct SplitGroup {
    static constexpr int SEG_BLOCKS = kWaves * TW * 32;
    static constexpr int PF = 2 * TW + 1;  // units of each lane loaded a segment ahead
    enum Table { kNone, kTwo, kThree };

    unsigned char *lds;
    F16x2Layout lay;
    const float *b;
    int K, m_hi;
    int sx, sb, T;
    bool always3;
    float doubt;  // scaled outputs below it may hang on the taps below 2^-14; or 0
    bool zeros;   // the segment last measured
    Table table;

    __device__ __forceinline__ int *words() const
    {
        return reinterpret_cast<int *>(lds + lay.words_offset);
    }
    __device__ __forceinline__ int units() const { return SEG_BLOCKS * 4 + 2 * m_hi; }

    __device__ __forceinline__ void build_two()
    {
        int unused = 0;
        build_tap_table<2, TW>(lds, lay.tab_offset, lay.copy2, b, K, m_hi, unused,
                               split_scale(sb));
        table = kTwo;
    }

    // Notes the magnitudes of the segment in `raw` in this wave's words, for
    // the scale and the choice that every wave makes after the next barrier.
    __device__ __forceinline__ void measure(const f32x4 (&raw)[PF][2], int tid)
    {
        float largest = 0.0f, least = __builtin_inff();  // NaN once there is one
        const int n = units();
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            if (tid + j * kThreads >= n) break;
#pragma unroll
            for (int c = 0; c < 8; c += 2) {
                largest = maximum3(largest, raw[j][c >> 2][c & 3], raw[j][c >> 2][(c & 3) + 1]);
                least = minimum3(least, raw[j][c >> 2][c & 3], raw[j][c >> 2][(c & 3) + 1]);
            }
        }
        const int wmx = wave_umax(abs_bits(largest));
        unsigned int wmn = (unsigned)wave_umin(abs_bits(least));
        if (wmn == 0) {  // the smallest nonzero one: zeros wrap round
            unsigned int mn = 0xffffffffu;
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                if (tid + j * kThreads >= n) break;
#pragma unroll
                for (int c = 0; c < 8; ++c) mn = min(mn, abs_bits(raw[j][c >> 2][c & 3]) - 1);
            }
            wmn = (unsigned)wave_umin(mn) + 1;
        }
        if ((tid & 63) == 0) {
            int *w = words() + (tid >> 6);
            w[kSampleMax] = wmx;
            w[kSampleExp] =
                wmn ? __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, wmn)) : 128;
        }
    }

    // Takes a filter and the first segment it is for (in `raw`).  The LDS is
    // free on entry and on return; barriers inside.
    __device__ __forceinline__ void begin(const float *taps, int ntaps, bool same_filter,
                                          const f32x4 (&raw)[PF][2])
    {
        // Opaque, so that nothing derived from it is kept in registers across
        // the work items of the ragged kernel.
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int wave = tid >> 6, lane = tid & 63;
        int *w = words();
        b = taps;
        K = ntaps;
        m_hi = mfma_m_hi(K);
        // Each thread takes a run of taps (K <= 9 * 256).
        constexpr int kRun = (kMaxTaps + kThreads - 1) / kThreads;
        const int run = (K + kThreads - 1) / kThreads;
        float v[kRun];
        if (!same_filter) {
            unsigned int m = 0;
#pragma unroll
            for (int r = 0; r < kRun; ++r) {
                const int k = tid * run + r;
                v[r] = r < run && k < K ? b[k] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < kRun; ++r) m = max(m, abs_bits(v[r]));
            m = (unsigned)wave_umax(m);
            if (lane == 0) w[kTapMax + wave] = (int)m;
        }
        measure(raw, tid);
        __syncthreads();
        if (same_filter) return;
        const unsigned int b_max = (unsigned)uniform(
            (int)max(max((unsigned)w[kTapMax], (unsigned)w[kTapMax + 1]),
                     max((unsigned)w[kTapMax + 2], (unsigned)w[kTapMax + 3])));
        sb = b_max < 0x7f800000u ? uniform(scale_exponent(b_max)) : 0;
        always3 = K < kMinTaps || b_max >= 0x7f800000u || sb < -100 || sb > 100;
        T = 10 + 31 - __builtin_clz(K + 1);
        doubt = 0.0f;
        table = kNone;
        if (always3) return;
        float err = 0.0f;
#pragma unroll
        for (int r = 0; r < kRun; ++r) {
            const float a = __builtin_fabsf(v[r] * pow2(sb));
            if (v[r] != 0.0f && a < 0x1p-14f) err += fmaxf(fminf(a, 0x1p-35f), 0x1p-149f);
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) err += __shfl_xor(err, d, 64);
        if (lane == 0) w[kTapErr + wave] = __builtin_bit_cast(int, err);
        build_two();
        __syncthreads();
        err = 0.0f;
        for (int i = 0; i < 4; ++i) err += __builtin_bit_cast(float, w[kTapErr + i]);
        // 2 err max|X| / ((K + 1) 2^-25), max|X| < 2^14.
        doubt = uniform(err * 0x1p+40f / (float)(K + 1));
    }

    // Whether the segment last measured fits the split, and its scale.
    __device__ __forceinline__ bool fit()
    {
        const int *w = words();
        const unsigned int mx = (unsigned)uniform((int)max(
            max((unsigned)w[0], (unsigned)w[1]), max((unsigned)w[2], (unsigned)w[3])));
        const int e = uniform(min(min(w[kSampleExp], w[kSampleExp + 1]),
                                  min(w[kSampleExp + 2], w[kSampleExp + 3])));
        sx = uniform(scale_exponent(mx));
        zeros = mx == 0;
        if (always3 || mx >= 0x7f800000u || sx < -100 || sx > 100) return false;
        return e >= 1 - T - sx;
    }

    // Half a segment's outputs (blocks P0 .. P0 + 127) by BF16x3.  Entered and
    // left with the LDS in use by no one after the next barrier.
    __device__ __forceinline__ void half_three(const float *__restrict__ xrow,
                                               float *__restrict__ yrow, int64_t N, int64_t P0,
                                               int wave, int lane)
    {
        const int tid = 64 * wave + lane;
        int *mins = words() + kMins3;
        __syncthreads();
        if (table != kThree) {
            int min_b = 0;
            build_tap_table<3, 1>(lds, lay.tab_offset, lay.copy3, b, K, m_hi, min_b);
            min_b = wave_min(min_b);
            if (lane == 0) mins[4 + wave] = min_b;
            table = kThree;
        }
        const int n = kWaves * 128 + 2 * m_hi;
        const int64_t xb = 32 * P0 - 16 * (int64_t)m_hi;
        int min_e = 0;
        for (int u = tid; u < n; u += kThreads) {
            f32x4 r[2];
            load_unit<REV>(xrow, N, xb, u, n, r);
            store_unit<3, 1, REV>(lds, lay.stride3, u, r, min_e);
        }
        min_e = wave_min(min_e);
        if (lane == 0) mins[wave] = min_e;
        __syncthreads();
        if (32 * (P0 + (int64_t)uniform(wave) * 32) < N) {
            const int i = lane & 31, g = lane >> 5;
            Contraction<3, 1> ct;
            contract_segment<3, 1>(ct, lds, lay.stride3, lay.tab_offset, lay.copy3, m_hi + 2,
                                   m_hi, wave, i, g);
            store_segment<3, 1, REV>(ct, yrow, N, P0, wave, i, g, xrow, b, K,
                                     segment_is_tiny(mins));
        }
    }

    // Filters the segment at block P0, whose units are in `raw` and measured
    // (a barrier since); `next()` loads the next segment's.  The LDS is free on
    // entry.
    template <class Next>
    __device__ __forceinline__ void segment(const f32x4 (&raw)[PF][2],
                                            const float *__restrict__ xrow,
                                            float *__restrict__ yrow, int64_t N, int64_t P0,
                                            int tid, Next next)
    {
        const int wave = tid >> 6, lane = tid & 63;
        const bool two = fit();
        if (two) {
            if (table != kTwo) build_two();
            const SplitScale scale = split_scale(sx);
            const int n = units();
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                const int u = tid + j * kThreads;
                if (u < n) store_unit2<TW, REV>(lds, lay.stride2, u, raw[j], scale);
            }
        }
        __syncthreads();
        next();
        if (two) {
            // A wave past the row end has no output (see fir_mfma_kernel).
            bool more = false;
            if (32 * (P0 + (int64_t)uniform(wave) * 32 * TW) < N) {
                const int i = lane & 31, g = lane >> 5;
                Contraction<2, TW> ct;
                contract_segment<2, TW>(ct, lds, lay.stride2, lay.tab_offset, lay.copy2,
                                        m_hi + 2, m_hi, wave, i, g);
                wait_for_loads();
                const int e = -(sx + sb);
                const float d = doubt > 0.0f && !zeros ? __builtin_ldexpf(doubt, e) + 0x1p-149f
                                                       : 0.0f;
                const SplitOutputs so = {e, d, m_hi};
                more = store_segment<2, TW, REV>(ct, yrow, N, P0, wave, i, g, xrow, b, K, false,
                                                 so);
            }
            if (doubt == 0.0f || zeros) return;
            int *w = words() + kRedo;
            const bool any = __any(more);
            if (lane == 0) w[wave] = any;
            __syncthreads();
            if (!uniform(w[0] | w[1] | w[2] | w[3])) return;
        }
#pragma unroll 1
        for (int h = 0; h < TW; ++h)
            if (32 * (P0 + 128 * h) < N) half_three(xrow, yrow, N, P0 + 128 * h, wave, lane);
    }
};

// One workgroup (4 waves) filters segs_per_wg consecutive segments, as
// fir_mfma_kernel does.
template <int TW, bool REV>
__global__ __launch_bounds__(kThreads, 2) void fir_f16x2_kernel(
    const float *__restrict__ x, int64_t ldx, int64_t N, float *__restrict__ y, int64_t ldy,
    const float *__restrict__ b, int K, int m_hi, int64_t row0, int segs_per_row, int64_t nsegs,
    int segs_per_wg, int64_t nwg, F16x2Layout lay)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    using Group = SplitGroup<TW, REV>;
    const int64_t seg_first = xcd_remap(blockIdx.x, nwg) * segs_per_wg;
    const int count = (int)min((int64_t)segs_per_wg, nsegs - seg_first);
    // Row and segment of the row, stepped: a 64-bit division is some 150
    // scalar instructions, and one stood before every contraction.
    const int64_t first_row = seg_first / segs_per_row;
    int seg = (int)(seg_first - first_row * segs_per_row);
    const float *xrow = x + (row0 + first_row) * ldx;
    float *yrow = y + (row0 + first_row) * ldy;
    f32x4 raw[Group::PF][2];
    auto prefetch = [&](const float *xr, int sg, int tid) {
        const int64_t xb = 32 * (int64_t)sg * Group::SEG_BLOCKS - 16 * (int64_t)m_hi;
#pragma unroll
        for (int j = 0; j < Group::PF; ++j)
            load_unit<REV>(xr, N, xb, tid + j * kThreads, Group::SEG_BLOCKS * 4 + 2 * m_hi,
                           raw[j]);
    };
    prefetch(xrow, seg, (int)threadIdx.x);
    Group group;
    group.lds = lds;
    group.lay = lay;
    group.begin(b, K, false, raw);
    for (int done = 0; done < count; ++done) {
        // Lane-dependent values are recomputed in every iteration (see
        // fir_mfma_kernel).
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int64_t P0 = (int64_t)seg * Group::SEG_BLOCKS;
        if (done) {
            group.measure(raw, tid);
            __syncthreads();  // the previous segment's MFMAs are done
        }
        const bool last = seg + 1 == segs_per_row;
        const int next_seg = last ? 0 : seg + 1;
        group.segment(raw, xrow, yrow, N, P0, tid, [&] {
            if (done + 1 < count) prefetch(last ? xrow + ldx : xrow, next_seg, tid);
        });
        seg = next_seg;
        if (last) {
            xrow += ldx;
            yrow += ldy;
        }
    }
}

// Ragged (CSR) batches: the work queue of fir_mfma_ragged_kernel.
constexpr int kRaggedTW = 2;
static_assert(kMfmaRaggedSegLen == 32 * kWaves * kRaggedTW * 32, "segment length");

__global__ __launch_bounds__(kThreads, 2) void fir_f16x2_ragged_kernel(
    const float *__restrict__ x, const float *__restrict__ b, float *__restrict__ y,
    const MfmaRaggedItem *__restrict__ items, int n_items, unsigned int *__restrict__ counter,
    F16x2Layout lay)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    using Group = SplitGroup<kRaggedTW, false>;
    // Two item slots, used in turn (see fir_mfma_ragged_kernel).
    int *s_item = reinterpret_cast<int *>(lds + lay.words_offset + 4 * kWords);
    f32x4 raw[Group::PF][2];
    auto prefetch = [&](const MfmaRaggedItem &q, int64_t sg, int tid) {
        const int mh = mfma_m_hi(q.K);
        const int64_t xb = 32 * sg * Group::SEG_BLOCKS - 16 * (int64_t)mh;
#pragma unroll
        for (int j = 0; j < Group::PF; ++j)
            load_unit<false>(x + q.x0, q.len, xb, tid + j * kThreads,
                             Group::SEG_BLOCKS * 4 + 2 * mh, raw[j]);
    };
    if (threadIdx.x == 0) s_item[0] = (int)atomicAdd(counter, 1u);
    __syncthreads();
    int nxt = uniform(s_item[0]);  // scalar, and the items with it
    if (nxt < n_items) prefetch(items[nxt], items[nxt].seg0, (int)threadIdx.x);
    Group group;
    group.lds = lds;
    group.lay = lay;
    group.b = nullptr;
    group.K = -1;
    for (int parity = 1;; parity ^= 1) {
        if (nxt >= n_items) break;  // uniform: read from LDS after a barrier
        const MfmaRaggedItem w = items[nxt];
        if (threadIdx.x == 0) s_item[parity] = (int)atomicAdd(counter, 1u);
        __syncthreads();  // every wave is done with the previous item's LDS; slot written
        nxt = uniform(s_item[parity]);
        group.begin(b + w.b0, w.K, b + w.b0 == group.b && w.K == group.K, raw);
        const int64_t seg_end = (int64_t)w.seg0 + w.nseg;
        for (int64_t sg = w.seg0; sg < seg_end; ++sg) {
            int tid = (int)threadIdx.x;
            asm volatile("" : "+v"(tid));
            const int64_t P0 = sg * Group::SEG_BLOCKS;
            if (sg != w.seg0) {
                group.measure(raw, tid);
                __syncthreads();  // the previous segment's MFMAs are done
            }
            group.segment(raw, x + w.x0, y + w.x0, w.len, P0, tid, [&] {
                if (sg + 1 < seg_end) {
                    prefetch(w, sg + 1, tid);
                } else if (nxt < n_items) {
                    prefetch(items[nxt], items[nxt].seg0, tid);
                }
            });
        }
    }
}

// Two workgroups share a CU's LDS (and the register file: 256 a lane).
constexpr size_t kHalfLds = kMaxLds / 2;

template <int TW, bool REV>
int launch_f16x2(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                 float *y, int64_t ldy, int segs_per_wg, hipStream_t stream)
{
    const F16x2Layout lay = f16x2_layout(K, TW);
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(&fir_f16x2_kernel<TW, REV>),
                               kMaxLds));
    const int64_t seg_len = 32 * (int64_t)SplitGroup<TW, REV>::SEG_BLOCKS;
    const int64_t segs = (N + seg_len - 1) / seg_len;
    if (segs > 0x7fffffff)
        return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "row too long (N=%lld)", (long long)N);
    const int64_t rows_per_launch = std::max<int64_t>(1, 0x7fffffff / segs);
    for (int64_t r0 = 0; r0 < B; r0 += rows_per_launch) {
        const int64_t nsegs = std::min(rows_per_launch, B - r0) * segs;
        const int64_t nwg = (nsegs + segs_per_wg - 1) / segs_per_wg;
        hipLaunchKernelGGL((fir_f16x2_kernel<TW, REV>), dim3((unsigned)nwg), dim3(kThreads),
                           f16x2_lds(lay), stream, x, ldx, N, y, ldy, b, K, mfma_m_hi(K), r0,
                           (int)segs, nsegs, segs_per_wg, nwg, lay);
        SCIR_TRY(check_launch("fir_f16x2_kernel"));
    }
    return SCIR_HIP_OK;
}

template <int TW>
int launch_f16x2_dir(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                     float *y, int64_t ldy, bool rev, int segs_per_wg, hipStream_t stream)
{
    return rev ? launch_f16x2<TW, true>(x, ldx, b, K, B, N, y, ldy, segs_per_wg, stream)
               : launch_f16x2<TW, false>(x, ldx, b, K, B, N, y, ldy, segs_per_wg, stream);
}

}  // namespace

bool fir_f16x2_takes(int K)
{
    return K >= 1 && K <= kMaxTaps && f16x2_lds(f16x2_layout(K, 2)) <= kHalfLds;
}

int fir_f16x2_dev(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                  float *y, int64_t ldy, bool rev, int64_t batch_rows, hipStream_t stream,
                  DeviceState *st)
{
    if (B == 0 || N == 0) return SCIR_HIP_OK;
    if (K == 0) return fill_zero_2d(y, ldy, B, N, stream);
    const TuneChoice tc = tune_lookup(K, N);
    // Segments of 8192 samples once two workgroups a CU have one ([64, 65536],
    // K = 129: 14.2 us against 17.0 with 4096), of 4096 for fewer or shorter
    // rows ([64, 16384], K = 512: 10.2 against 12.8).
    const int64_t long_segs = batch_rows * ((N + kMfmaRaggedSegLen - 1) / kMfmaRaggedSegLen);
    const int tw = N <= 4096 || long_segs < 2 * (int64_t)st->cu_count ? 1 : 2;
    const int64_t seg_len = 32 * (int64_t)kWaves * tw * 32;
    const int64_t total = B * ((N + seg_len - 1) / seg_len);
    const int64_t cap = tc.mfma_segs_forced
                            ? total
                            : std::max<int64_t>(1, total / (4 * (int64_t)std::max(1, st->cu_count)));
    const int spw = (int)std::max<int64_t>(1, std::min<int64_t>(tc.mfma_segs, cap));
    return tw == 1 ? launch_f16x2_dir<1>(x, ldx, b, K, B, N, y, ldy, rev, spw, stream)
                   : launch_f16x2_dir<2>(x, ldx, b, K, B, N, y, ldy, rev, spw, stream);
}

int fir_f16x2_ragged_occupancy(int kmax, size_t *lds, int *per_cu)
{
    *lds = f16x2_lds(f16x2_layout(std::max(kmax, 1), kRaggedTW));
    const void *fn = reinterpret_cast<const void *>(&fir_f16x2_ragged_kernel);
    int n = 0;
    SCIR_TRY(allow_dynamic_lds(fn, kMaxLds));
    SCIR_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kThreads, *lds));
    *per_cu = std::max(1, n);
    return SCIR_HIP_OK;
}

int fir_f16x2_ragged_launch(const float *x, const float *b, float *y, const MfmaRaggedItem *items,
                            int n_items, unsigned int *counter, int kmax, size_t lds, int grid,
                            hipStream_t stream)
{
    const F16x2Layout lay = f16x2_layout(std::max(kmax, 1), kRaggedTW);
    if (f16x2_lds(lay) != lds)
        return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "ragged F16x2 layout mismatch");
    SCIR_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(&fir_f16x2_ragged_kernel), kMaxLds));
    hipLaunchKernelGGL(fir_f16x2_ragged_kernel, dim3((unsigned)grid), dim3(kThreads), lds, stream,
                       x, b, y, items, n_items, counter, lay);
    return check_launch("fir_f16x2_ragged_kernel");
}

}  // namespace scir
