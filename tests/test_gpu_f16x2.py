"""F32 by two fp16 terms (fir_f16x2.hip): every output within F32's bound,
(K+1) 2^-23 sum|b||x| of the FP64 oracle (plus one subnormal unit a term),
where the kernel can go wrong: segment edges, the largest filter, filters
short enough to run by BF16x3 beside longer ones, both directions, samples of
every magnitude, magnitudes that fp16 cannot hold together, and filters with
taps that are almost zero meeting samples that are zero."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


def bound(oracle, x, b):
    return oracle.fir_error_bound(x, b) + (b.size + 1) * 2.0 ** -149


def check(oracle, x, b, what):
    """Forward and back to front on the device, against the oracle."""
    import torch
    from scir_amd import device
    print(f"f16x2 {what} x{x.shape} K={b.size}", flush=True)
    xt, bt = torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda")
    y = device.fir(xt, bt, "f32").cpu().numpy().astype(np.float64)
    excess = np.abs(y - oracle.lfilter_f64(x, b)) - bound(oracle, x, b)
    assert np.all(excess <= 0), f"{what}: excess {excess.max()} at {np.argmax(excess)}"
    dx = device.vjp_dx(xt, bt, "f32").cpu().numpy().astype(np.float64)
    xr = np.ascontiguousarray(x[:, ::-1])
    excess = np.abs(dx[:, ::-1] - oracle.lfilter_f64(xr, b)) - bound(oracle, xr, b)
    assert np.all(excess <= 0), f"{what} back to front: excess {excess.max()}"


# Filters above 513 taps take this path at any size: the shortest of them, the
# longest (2049: the history fills the units loaded ahead), and the next.
@pytest.mark.parametrize("K", [514, 1023, 2049, 2050])
@pytest.mark.parametrize("N", [1, 31, 4095, 4096, 4097, 8191, 8193, 20000])
def test_segment_edges(hip, oracle, K, N):
    r = rng(K * 7 + N)
    x = r.standard_normal((3, N)).astype(np.float32)
    x[1, ::53] *= 1000.0
    check(oracle, x, r.standard_normal(K).astype(np.float32), "edges")


def sinc_with_zero_crossings(K):
    from scir_amd import design
    b = design.lowpass(K, 0.2)
    assert np.count_nonzero(np.abs(b) < 1e-9 * np.abs(b).max()) > K // 10
    return b


# Zero samples under taps that are almost zero: outputs that hang on one such
# tap (at the row start, between impulses), silent stretches, zero rows.
@pytest.mark.parametrize("K", [601, 1023])
@pytest.mark.parametrize("what", ["quantised", "edges", "sparse", "zero_rows"])
def test_zero_samples_and_almost_zero_taps(hip, oracle, K, what):
    r = rng(K + len(what))
    x = r.standard_normal((3, 20000)).astype(np.float32)
    if what == "quantised":
        x = np.round(x * 4).astype(np.float32)
    elif what == "edges":
        x[0, 300:9000] = 0.0
        x[1, :8192] = 0.0
        x[2, 4096:] = 0.0
    elif what == "sparse":
        x = np.where(np.arange(20000) % 2500 == 7, x, 0.0).astype(np.float32)
    else:
        x[:2] = 0.0
        x[2, 1:] = 0.0
    b = sinc_with_zero_crossings(K)
    b[0] = np.float32(3e-17)
    check(oracle, x, b, f"zeros {what}")


@pytest.mark.parametrize("case", ["1e-30", "1e30", "1e-41", "ramp", "bursts", "impulses",
                                  "silence", "steps", "near_max"])
@pytest.mark.parametrize("taps", ["random", "sinc", "decaying", "tiny"])
def test_magnitudes(hip, oracle, case, taps):
    r = rng(len(case) * 31 + len(taps))
    K, N = 601, 26000
    x = r.standard_normal((2, N)).astype(np.float32)
    if case in ("1e-30", "1e30", "1e-41"):
        x = (x.astype(np.float64) * float(case)).astype(np.float32)
    elif case == "ramp":  # forty orders of magnitude along the row
        x = (x * 10.0 ** np.linspace(-22, 18, N)).astype(np.float32)
    elif case == "bursts":  # loud samples in faint ones
        x = (x * np.where(r.random((2, N)) < 2e-3, 1e6, 1e-6)).astype(np.float32)
    elif case == "impulses":
        x = np.where(r.random((2, N)) < 1e-3, x, 0.0).astype(np.float32)
    elif case == "silence":
        x[:, :9000] = 0.0
        x[0, 15000:24000] = 0.0
    elif case == "steps":
        x = np.round(x * 3).astype(np.float32)
    elif case == "near_max":
        x[:, 12000:12010] *= np.float32(1e36)
    b = r.standard_normal(K).astype(np.float32)
    if taps == "sinc":
        b = sinc_with_zero_crossings(K)
    elif taps == "decaying":
        b = (b * 0.9 ** np.arange(K)).astype(np.float32)
    elif taps == "tiny":
        b = (b * 1e-30).astype(np.float32)
    check(oracle, x, b, f"{case}/{taps}")


def test_taken_from_its_size_up_matches_fp32_matrix_cores(hip, oracle):
    """At a size and length where F32 moves from the FP32 matrix cores to this
    path both stay within the bound, and they are not the same numbers."""
    import torch
    from scir_amd import device
    L = hip.lib()
    r = rng(5)
    x = r.standard_normal((40, 65537)).astype(np.float32)
    b = sinc_with_zero_crossings(255)
    xt, bt = torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda")
    y = device.fir(xt, bt, "f32").cpu().numpy()
    try:
        hip.check(L.scir_hip_tune_set(b"direct.mfma_strip", 8))
        y32 = device.fir(xt, bt, "f32").cpu().numpy()
    finally:
        hip.check(L.scir_hip_tune_set(b"direct.mfma_strip", -1))
    assert not np.array_equal(y, y32)
    y64, lim = oracle.lfilter_f64(x, b), bound(oracle, x, b)
    assert np.all(np.abs(y - y64) <= lim) and np.all(np.abs(y32 - y64) <= lim)


@pytest.mark.parametrize("K,precision", [(1023, "f32"), (300, "auto"), (2100, "f32")])
def test_parts_of_a_batch_run_by_its_arithmetic(hip, K, precision):
    """A batch that the host tier takes in parts of one row: the bits of the
    whole on the device, where a row by itself would run another way."""
    import torch
    from scir_amd import device
    L = hip.lib()
    r = rng(K)
    x = r.standard_normal((70, 65536)).astype(np.float32)
    b = r.standard_normal(K).astype(np.float32)
    print(f"f16x2 parts {precision} K={K}", flush=True)
    want = device.fir(torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda"), precision)
    y = np.empty_like(x)
    hip.check(L.scir_hip_tune_set(b"host.chunk_kib", 256))
    try:
        hip.check(L.scir_hip_fir_f32_host(
            x.ctypes.data, x.shape[1], b.ctypes.data, K, *x.shape, y.ctypes.data, x.shape[1],
            hip.precision_code(precision)))
    finally:
        hip.check(L.scir_hip_tune_set(b"host.chunk_kib", -1))
    assert np.array_equal(y, want.cpu().numpy())


def test_long_segments_of_many_rows(hip, oracle):
    """Rows enough that the segments are of 8192 samples (test_segment_edges
    has the short ones): one, and one sample into the second."""
    import torch
    from scir_amd import device
    r = rng(8)
    for rows, N in ((513, 8192), (300, 8193)):
        print(f"f16x2 long segments [{rows},{N}]", flush=True)
        x = r.standard_normal((rows, N)).astype(np.float32)
        b = r.standard_normal(514).astype(np.float32)
        y = device.fir(torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda"), "f32")
        keep = [0, 1, rows // 2, rows - 1]
        y = y.cpu().numpy()[keep].astype(np.float64)
        assert np.all(np.abs(y - oracle.lfilter_f64(x[keep], b)) <= bound(oracle, x[keep], b))


def test_ragged_filters_of_every_length(hip, oracle):
    """One batch with filters from 0 to 1500 taps (below 16: BF16x3), with
    the work (a long signal) that makes its F32 plan take this path."""
    import torch
    from scir_amd.ragged import RaggedPlan
    r = rng(77)
    ks = np.array([0, 1, 2, 7, 15, 16, 17, 32, 33, 64, 200, 513, 1500, 1500, 3, 900])
    lens = np.array([100, 5, 9000, 8192, 8193, 1, 4096, 20000, 3, 100, 7000, 16385, 130000, 0, 0,
                     2500])
    assert np.sum(lens * ks) > 1.9e8
    offs = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
    boffs = np.concatenate(([0], np.cumsum(ks))).astype(np.int64)
    x = r.standard_normal(int(offs[-1])).astype(np.float32)
    b = r.standard_normal(int(boffs[-1])).astype(np.float32)
    print("f16x2 ragged lengths", flush=True)
    plan = RaggedPlan(offs, boffs, "f32")
    y = plan.execute(torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda"))
    y = y.cpu().numpy()
    plan.close()
    y64 = oracle.lfilter_ragged_f64(x, offs, b, boffs)
    for s in range(lens.size):
        seg = slice(offs[s], offs[s + 1])
        taps = b[boffs[s]:boffs[s + 1]]
        lim = bound(oracle, x[seg], taps)[0] if taps.size and lens[s] else 0.0
        assert np.all(np.abs(y[seg] - y64[seg]) <= lim), f"signal {s}: {lens[s]}, K={ks[s]}"
