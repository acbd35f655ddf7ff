// Long-tap batched FIR as a Toeplitz-block contraction on gfx950 MFMA
// (v_mfma_f32_32x32x16_{bf16,f16}), FP32 accumulation.
//
// The contraction (operand layout, split terms, epilogue) is in
// toeplitz_mfma.hpp; here are the dense and the ragged kernel of BF16x3 and
// FP16 and their launches.
#include "toeplitz_mfma.hpp"

namespace scir {
namespace {

// One workgroup (4 waves) computes segs_per_wg consecutive segments of
// kWaves*TW*32 output blocks each (segment id = row * segs_per_row + index in
// the row).  A segment needs LDS units 0 .. units-1: 2*m_hi units of history
// and 4*SEG_BLOCKS of its own samples.  The first PF = 2*TW + 1 units of
// each lane (unit lane + 256*j) are loaded into registers one segment ahead:
// they are in flight while the waves run the previous segment's MFMAs.
// Units past PF*256 (only when 2*m_hi > 256) are loaded when the segment is
// staged.
template <int S, int TW, bool REV>
__global__ __launch_bounds__(kThreads) void fir_mfma_kernel(
    const float *__restrict__ x, int64_t ldx, int64_t N, float *__restrict__ y, int64_t ldy,
    const float *__restrict__ b, int K, int msteps, int m_hi, int64_t row0, int segs_per_row,
    int64_t nsegs, int segs_per_wg, int64_t nwg, int split_stride, int tab_offset,
    int copy_bytes)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int SEG_BLOCKS = kWaves * TW * 32;
    constexpr int PF = 2 * TW + 1;
    const int64_t lid = xcd_remap(blockIdx.x, nwg);
    const int64_t seg_first = lid * segs_per_wg;
    const int count = (int)min((int64_t)segs_per_wg, nsegs - seg_first);
    const int units = SEG_BLOCKS * 4 + 2 * m_hi;
    // Row and segment of the row, stepped: a 64-bit division is some 150
    // scalar instructions, and one stood before every contraction.
    const int64_t first_row = seg_first / segs_per_row;
    int seg = (int)(seg_first - first_row * segs_per_row);
    const float *xrow = x + (row0 + first_row) * ldx;
    float *yrow = y + (row0 + first_row) * ldy;

    f32x4 raw[PF][2];
    // Sample index of LDS unit 0 of a row's segment sg.
    auto first_sample = [&](int sg) { return 32 * (int64_t)sg * SEG_BLOCKS - 16 * (int64_t)m_hi; };
    auto prefetch = [&](const float *xr, int sg, int tid) {
#pragma unroll
        for (int j = 0; j < PF; ++j)
            load_unit<REV>(xr, N, first_sample(sg), tid + j * kThreads, units, raw[j]);
    };
    prefetch(xrow, seg, (int)threadIdx.x);

    // Tap tables, built while the first segment's loads are in flight.
    int *mins = reinterpret_cast<int *>(lds + tab_offset + 2 * S * copy_bytes);
    {
        int min_b = 0;
        build_tap_table<S, TW>(lds, tab_offset, copy_bytes, b, K, m_hi, min_b);
        if (S == 3) {
            min_b = wave_min(min_b);
            if ((threadIdx.x & 63) == 0) mins[4 + (threadIdx.x >> 6)] = min_b;
        }
    }

    for (int done = 0; done < count; ++done) {
        // Lane-dependent values are recomputed in every iteration rather than
        // hoisted out of the loop, where they would hold registers through
        // the contraction.
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int wave = tid >> 6, lane = tid & 63;
        const int i = lane & 31, g = lane >> 5;
        const int64_t P0 = (int64_t)seg * SEG_BLOCKS, xb = first_sample(seg);
        const bool last = seg + 1 == segs_per_row;
        const int next_seg = last ? 0 : seg + 1;

        // ---- stage: x[xb .. xb + 8*units) -> S split arrays in LDS ----
        if (done) __syncthreads();  // the previous segment's MFMAs are done
        int min_e = 0;
        stage_segment<S, TW, PF, REV>(lds, split_stride, raw, xrow, N, xb, units, tid, min_e);
        if (S == 3) {
            const int m = wave_min(min_e);
            if (lane == 0) mins[wave] = m;
        }
        __syncthreads();
        if (done + 1 < count) prefetch(last ? xrow + ldx : xrow, next_seg, tid);

        // ---- contraction and epilogue ----
        // Wave w's tiles cover outputs 32*(P0 + 32*TW*w) .. +1024*TW-1 of the
        // row: a wave past the row end has no output and skips both (the
        // contraction has no barrier), leaving the SIMD's matrix pipe to the
        // other wave on it.
        if (32 * (P0 + (int64_t)__builtin_amdgcn_readfirstlane(wave) * 32 * TW) < N) {
            Contraction<S, TW> ct;
            contract_segment<S, TW>(ct, lds, split_stride, tab_offset, copy_bytes, msteps, m_hi,
                                    wave, i, g);
            wait_for_loads();
            // Read after the contraction (the words change only after the
            // next segment's first barrier): nothing extra stays live through it.
            const bool tiny = S == 3 && segment_is_tiny(mins);
            store_segment<S, TW, REV>(ct, yrow, N, P0, wave, i, g, xrow, b, K, tiny);
        }
        seg = next_seg;
        if (last) {
            xrow += ldx;
            yrow += ldy;
        }
    }
}

// Ragged (CSR) batches: a persistent grid pulls work items (a run of
// consecutive segments of one signal, longest first) through an atomic
// counter until the queue is drained; every workgroup leaves the loop on its
// first fetch past the end.  Each segment is staged, contracted and stored as
// in the dense kernel, with the item's own taps and length; the tap tables are
// rebuilt only when the item's taps differ from the ones in LDS.  Items are
// claimed one ahead and broadcast through the 16 bytes of LDS at
// `slot_offset`; the next item's first segment loads during the current
// item's last contraction.
template <int S, int TW>
__global__ __launch_bounds__(kThreads) void fir_mfma_ragged_kernel(
    const float *__restrict__ x, const float *__restrict__ b, float *__restrict__ y,
    const MfmaRaggedItem *__restrict__ items, int n_items, unsigned int *__restrict__ counter,
    int split_stride, int tab_offset, int copy_bytes, int slot_offset)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int SEG_BLOCKS = kWaves * TW * 32;
    constexpr int PF = 2 * TW + 1;
    // Two item slots, used in turn: the index claimed at the start of item n
    // is read by every lane right after that item's first barrier, and the
    // slot is written again two items later, after the next item's barrier.
    int *s_item = reinterpret_cast<int *>(lds + slot_offset);
    int *mins = reinterpret_cast<int *>(lds + slot_offset + 16);
    int64_t tab_b0 = -1;
    int tab_K = -1;
    f32x4 raw[PF][2];
    // The first segment of item q, into raw (also for the next item, during
    // the current item's last contraction).
    auto prefetch = [&](const MfmaRaggedItem &q, int64_t sg, int tid) {
        const int mh = mfma_m_hi(q.K);
        const int64_t xb = 32 * sg * SEG_BLOCKS - 16 * (int64_t)mh;
#pragma unroll
        for (int j = 0; j < PF; ++j)
            load_unit<false>(x + q.x0, q.len, xb, tid + j * kThreads, SEG_BLOCKS * 4 + 2 * mh,
                             raw[j]);
    };
    if (threadIdx.x == 0) s_item[0] = (int)atomicAdd(counter, 1u);
    __syncthreads();
    int nxt = s_item[0];
    MfmaRaggedItem wn{};
    if (nxt < n_items) {
        wn = items[nxt];
        prefetch(wn, wn.seg0, (int)threadIdx.x);
    }
    for (int parity = 1;; parity ^= 1) {
        const int it = nxt;
        if (it >= n_items) break;  // uniform: read from LDS after a barrier
        const MfmaRaggedItem w = wn;
        // Claim the item after this one now, so its first segment can load
        // during this item's last contraction.
        if (threadIdx.x == 0) s_item[parity] = (int)atomicAdd(counter, 1u);
        __syncthreads();  // every wave is done with the previous item's LDS; slot written
        nxt = s_item[parity];
        const int m_hi = mfma_m_hi(w.K), msteps = m_hi + 2;
        const int units = SEG_BLOCKS * 4 + 2 * m_hi;
        const float *__restrict__ xrow = x + w.x0;
        float *__restrict__ yrow = y + w.x0;
        const int64_t seg_end = (int64_t)w.seg0 + w.nseg;
        if (w.b0 != tab_b0 || w.K != tab_K) {
            int min_b = 0;
            build_tap_table<S, TW>(lds, tab_offset, copy_bytes, b + w.b0, w.K, m_hi, min_b);
            if (S == 3) {
                min_b = wave_min(min_b);
                if ((threadIdx.x & 63) == 0) mins[4 + (threadIdx.x >> 6)] = min_b;
            }
            tab_b0 = w.b0;
            tab_K = w.K;
        }
        for (int64_t sg = w.seg0; sg < seg_end; ++sg) {
            int tid = (int)threadIdx.x;
            asm volatile("" : "+v"(tid));
            const int wave = tid >> 6, lane = tid & 63;
            const int i = lane & 31, g = lane >> 5;
            const int64_t P0 = sg * SEG_BLOCKS;
            const int64_t xb = 32 * P0 - 16 * (int64_t)m_hi;
            if (sg != w.seg0) __syncthreads();  // the previous segment's MFMAs are done
            int min_e = 0;
            stage_segment<S, TW, PF, false>(lds, split_stride, raw, xrow, w.len, xb, units, tid,
                                            min_e);
            if (S == 3) {
                const int m = wave_min(min_e);
                if (lane == 0) mins[wave] = m;
            }
            __syncthreads();
            if (sg + 1 < seg_end) {
                prefetch(w, sg + 1, tid);
            } else if (nxt < n_items) {
                wn = items[nxt];
                prefetch(wn, wn.seg0, tid);
            }
            // A wave whose outputs all lie past the signal's end skips its
            // contraction and epilogue (as in the dense kernel).
            if (32 * (P0 + (int64_t)__builtin_amdgcn_readfirstlane(wave) * 32 * TW) < w.len) {
                Contraction<S, TW> ct;
                contract_segment<S, TW>(ct, lds, split_stride, tab_offset, copy_bytes, msteps,
                                        m_hi, wave, i, g);
                wait_for_loads();
                const bool tiny = S == 3 && segment_is_tiny(mins);
                store_segment<S, TW, false>(ct, yrow, w.len, P0, wave, i, g, xrow, b + w.b0,
                                            w.K, tiny);
            }
        }
    }
}

constexpr int kRaggedTW = 2;
static_assert(kMfmaRaggedSegLen == 32 * kWaves * kRaggedTW * 32, "segment length");

template <int S, int TW>
size_t mfma_lds_bytes(int K)
{
    const int m_hi = mfma_m_hi(K);
    const int units = kWaves * TW * 32 * 4 + 2 * m_hi;
    return (size_t)S * unit_bytes(units, TW) + (size_t)2 * S * tab_copy_bytes(m_hi, TW) +
           kMinsBytes;
}

template <int S, int TW, bool REV>
int launch_mfma_dir(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                    float *y, int64_t ldy, int segs_per_wg, hipStream_t stream)
{
    constexpr int SEG_BLOCKS = kWaves * TW * 32;
    const int m_hi = mfma_m_hi(K), msteps = mfma_steps(K);
    const int units = SEG_BLOCKS * 4 + 2 * m_hi;
    const int split_stride = (int)unit_bytes(units, TW);
    const int tab_offset = S * split_stride;
    const int copy_bytes = tab_copy_bytes(m_hi, TW);
    const size_t lds = mfma_lds_bytes<S, TW>(K);
    SCIR_TRY(
        allow_dynamic_lds(reinterpret_cast<const void *>(&fir_mfma_kernel<S, TW, REV>), kMaxLds));
    const int64_t seg_len = 32 * (int64_t)SEG_BLOCKS;
    const int64_t segs = (N + seg_len - 1) / seg_len;
    if (segs > 0x7fffffff)
        return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "row too long (N=%lld)", (long long)N);
    const int64_t rows_per_launch = std::max<int64_t>(1, 0x7fffffff / segs);
    for (int64_t r0 = 0; r0 < B; r0 += rows_per_launch) {
        const int64_t rows = std::min(rows_per_launch, B - r0);
        const int64_t nsegs = rows * segs;
        const int64_t nwg = (nsegs + segs_per_wg - 1) / segs_per_wg;
        hipLaunchKernelGGL((fir_mfma_kernel<S, TW, REV>), dim3((unsigned)nwg), dim3(kThreads),
                           lds, stream, x, ldx, N, y, ldy, b, K, msteps, m_hi, r0, (int)segs,
                           nsegs, segs_per_wg, nwg, split_stride, tab_offset, copy_bytes);
        SCIR_TRY(check_launch("fir_mfma_kernel"));
    }
    return SCIR_HIP_OK;
}

// The direction is a template argument: a run-time flag puts a join after
// every prefetch load, at which the compiler waits for the loads in flight.
template <int S, int TW>
int launch_mfma(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                float *y, int64_t ldy, bool rev, int segs_per_wg, hipStream_t stream)
{
    return rev ? launch_mfma_dir<S, TW, true>(x, ldx, b, K, B, N, y, ldy, segs_per_wg, stream)
               : launch_mfma_dir<S, TW, false>(x, ldx, b, K, B, N, y, ldy, segs_per_wg, stream);
}

template <int S>
int run_mfma(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N, float *y,
             int64_t ldy, bool rev, hipStream_t stream, const DeviceState *st)
{
    const TuneChoice tc = tune_lookup(K, N);
    int tw = S == 3 ? tc.mfma_tiles : tc.mfma_tiles_fp16;
    // Short rows: smaller segments keep the grid full.
    if (N <= 4096) tw = 1;
    // Long filters: fewer tiles per wave when the LDS would overflow.
    if (tw >= 4 && mfma_lds_bytes<S, 4>(K) > (size_t)kMaxLds) tw = 2;
    if (tw >= 2 && mfma_lds_bytes<S, 2>(K) > (size_t)kMaxLds) tw = 1;
    if (mfma_lds_bytes<S, 1>(K) > (size_t)kMaxLds)
        return fail(SCIR_HIP_ERR_UNSUPPORTED, "K=%d needs more LDS than the MFMA path has", K);
    // Segments per workgroup: as tuned, but (unless forced) never so many
    // that fewer than four workgroups per CU remain.
    const int64_t seg_len = 32 * (int64_t)kWaves * tw * 32;
    const int64_t total = B * ((N + seg_len - 1) / seg_len);
    const int64_t cap = tc.mfma_segs_forced
                            ? total
                            : std::max<int64_t>(1, total / (4 * (int64_t)std::max(1, st->cu_count)));
    const int spw = (int)std::max<int64_t>(1, std::min<int64_t>(tc.mfma_segs, cap));
    switch (tw) {
    case 1: return launch_mfma<S, 1>(x, ldx, b, K, B, N, y, ldy, rev, spw, stream);
    case 4: return launch_mfma<S, 4>(x, ldx, b, K, B, N, y, ldy, rev, spw, stream);
    default: return launch_mfma<S, 2>(x, ldx, b, K, B, N, y, ldy, rev, spw, stream);
    }
}

}  // namespace

bool fir_mfma_takes(int precision, int K)
{
    if (K <= 0) return true;
    const size_t need = precision == SCIR_HIP_PREC_BF16X3 ? mfma_lds_bytes<3, 1>(K)
                                                          : mfma_lds_bytes<1, 1>(K);
    return need <= (size_t)kMaxLds;
}

int fir_mfma_dev(const float *x, int64_t ldx, const float *b, int K, int64_t B, int64_t N,
                 float *y, int64_t ldy, int precision, bool rev, hipStream_t stream,
                 DeviceState *st)
{
    if (B == 0 || N == 0) return SCIR_HIP_OK;
    if (K == 0) return fill_zero_2d(y, ldy, B, N, stream);
    if (precision == SCIR_HIP_PREC_BF16X3)
        return run_mfma<3>(x, ldx, b, K, B, N, y, ldy, rev, stream, st);
    if (precision == SCIR_HIP_PREC_FP16)
        return run_mfma<1>(x, ldx, b, K, B, N, y, ldy, rev, stream, st);
    return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "precision %d is not an MFMA mode", precision);
}

namespace {

// Ragged LDS layout: S split arrays, the tap tables, then the item slot.
template <int S>
struct RaggedLayout {
    int split_stride, tab_offset, copy_bytes, slot_offset;
    size_t bytes;
    explicit RaggedLayout(int kmax)
    {
        const int m_hi = mfma_m_hi(kmax);
        const int units = kWaves * kRaggedTW * 32 * 4 + 2 * m_hi;
        split_stride = (int)unit_bytes(units, kRaggedTW);
        tab_offset = S * split_stride;
        copy_bytes = tab_copy_bytes(m_hi, kRaggedTW);
        slot_offset = tab_offset + 2 * S * copy_bytes;
        bytes = (size_t)slot_offset + 16 + kMinsBytes;
    }
};

template <int S>
int ragged_launch(const float *x, const float *b, float *y, const MfmaRaggedItem *items,
                  int n_items, unsigned int *counter, int kmax, size_t lds, int grid,
                  hipStream_t stream)
{
    const RaggedLayout<S> lay(kmax);
    if (lay.bytes != lds || lds > (size_t)kMaxLds)
        return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "ragged MFMA layout mismatch");
    SCIR_TRY(allow_dynamic_lds(
        reinterpret_cast<const void *>(&fir_mfma_ragged_kernel<S, kRaggedTW>), kMaxLds));
    hipLaunchKernelGGL((fir_mfma_ragged_kernel<S, kRaggedTW>), dim3((unsigned)grid),
                       dim3(kThreads), lds, stream, x, b, y, items, n_items, counter,
                       lay.split_stride, lay.tab_offset, lay.copy_bytes, lay.slot_offset);
    return check_launch("fir_mfma_ragged_kernel");
}

}  // namespace

int fir_mfma_ragged_lds(int precision, int kmax, size_t *lds)
{
    const size_t bytes = precision == SCIR_HIP_PREC_BF16X3 ? RaggedLayout<3>(kmax).bytes
                                                           : RaggedLayout<1>(kmax).bytes;
    if (bytes > (size_t)kMaxLds)
        return fail(SCIR_HIP_ERR_UNSUPPORTED,
                    "ragged MFMA batches take taps up to the LDS limit; K=%d needs %zu bytes",
                    kmax, bytes);
    *lds = bytes;
    return SCIR_HIP_OK;
}

int fir_mfma_ragged_occupancy(int precision, size_t lds, int *per_cu)
{
    int n = 0;
    const void *fn = precision == SCIR_HIP_PREC_BF16X3
                         ? reinterpret_cast<const void *>(&fir_mfma_ragged_kernel<3, kRaggedTW>)
                         : reinterpret_cast<const void *>(&fir_mfma_ragged_kernel<1, kRaggedTW>);
    SCIR_TRY(allow_dynamic_lds(fn, kMaxLds));
    SCIR_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kThreads, lds));
    *per_cu = std::max(1, n);
    return SCIR_HIP_OK;
}

int fir_mfma_ragged_launch(const float *x, const float *b, float *y, const MfmaRaggedItem *items,
                           int n_items, unsigned int *counter, int precision, int kmax,
                           size_t lds, int grid, hipStream_t stream)
{
    if (precision == SCIR_HIP_PREC_BF16X3)
        return ragged_launch<3>(x, b, y, items, n_items, counter, kmax, lds, grid, stream);
    if (precision == SCIR_HIP_PREC_FP16)
        return ragged_launch<1>(x, b, y, items, n_items, counter, kmax, lds, grid, stream);
    return fail(SCIR_HIP_ERR_INVALID_ARGUMENT, "precision %d is not an MFMA mode", precision);
}

}  // namespace scir
