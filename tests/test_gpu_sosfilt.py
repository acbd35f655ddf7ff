"""sosfilt / filtfilt on the GPU against the oracle (the reference loop).

reference_order (and rows of at most 1024 samples): every output equal to
the reference loop bit for bit.  Parallel in time (default): the first 16
outputs of each row bit for bit (they run from the zero start state like the
reference), and every output within 1e-12 of the row's largest |y| of the
reference loop (the joins carry the rounding of the state transitions;
measured ~1e-15).  Ill-conditioned cascades (high-order Chebyshev) make the
reference loop itself err by more than that: then both are compared with an
extended-precision run, and the GPU's error may be at most 16 times the
reference loop's (plus 1e-14 of the row's largest |y|)."""
import pathlib

import numpy as np
import pytest
import torch
from scipy import signal as ss

from oracle import oracle as orc
from scir_amd import device, signal
from scir_amd.gpu import Device

pytestmark = pytest.mark.gpu
GOLD = pathlib.Path(__file__).resolve().parent / "golden"
REL_TOL = 1e-12


def _sos(S, seed=0):
    if S == 0:
        return np.zeros((0, 6))
    base = [ss.butter(2 * S, 0.15, output="sos"),
            ss.cheby1(2 * S, 0.5, 0.3, output="sos"),
            ss.butter(S, [0.1, 0.35], "bandpass", output="sos")[:S]]
    return np.ascontiguousarray(base[seed % 3][:S])


def _check(y, ref, exact_prefix, sos=None, x=None, zero_phase=False):
    assert y.shape == ref.shape
    if exact_prefix:
        k = min(16, ref.shape[1])
        assert np.array_equal(y[:, :k], ref[:, :k])
    scale = np.max(np.abs(ref), axis=1, keepdims=True) + 1e-300
    err = np.max(np.abs(y - ref) / scale)
    if err <= REL_TOL:
        return
    assert sos is not None, err
    exact = orc.sosfilt_longdouble(sos, x, zero_phase).astype(np.float64)
    err_gpu = np.max(np.abs(y - exact) / scale)
    err_ref = np.max(np.abs(ref - exact) / scale)
    assert err_gpu <= 16 * err_ref + 1e-14, (err_gpu, err_ref)


@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16])
@pytest.mark.parametrize("shape", [(3, 1), (2, 17), (4, 1000), (3, 4133), (1, 70001)])
def test_reference_order_bitwise(S, shape):
    print(f"sosfilt reference_order S={S} shape={shape}", flush=True)
    rng = np.random.default_rng(S * 7 + shape[1])
    x = rng.standard_normal(shape)
    sos = _sos(S, S)
    y = signal.sosfilt_batched(sos, x, Device.Hip, reference_order=True)
    assert np.array_equal(y, orc.sosfilt_f64(sos, x))
    yf = signal.filtfilt_batched(sos, x, Device.Hip, reference_order=True)
    assert np.array_equal(yf, orc.filtfilt_f64(sos, x))


@pytest.mark.parametrize("S", [1, 2, 3, 4, 8, 9, 16])
@pytest.mark.parametrize("shape", [(2, 17), (4, 1000), (3, 4133), (1, 70001), (64, 9000)])
def test_chunked_close(S, shape):
    print(f"sosfilt chunked S={S} shape={shape}", flush=True)
    rng = np.random.default_rng(S * 11 + shape[1])
    x = rng.standard_normal(shape)
    sos = _sos(S, S + 1)
    _check(signal.sosfilt_batched(sos, x, Device.Hip), orc.sosfilt_f64(sos, x), True, sos, x)
    _check(signal.filtfilt_batched(sos, x, Device.Hip), orc.filtfilt_f64(sos, x), False, sos, x,
           zero_phase=True)


@pytest.mark.parametrize("design", ["low_pass", "high_pass", "band_pass", "band_stop"])
def test_reference_iir_fixtures(design):
    # the reference's own DF2T fixtures at its tolerance (1e-12 absolute)
    x = np.load(GOLD / "iir_bridge.npy")[1]
    sos = np.load(GOLD / f"iir_{design}_sos.npy")
    want = np.load(GOLD / f"iir_{design}_expected.npy")
    for ref_order in (False, True):
        y = signal.sosfilt_batched(sos, x[None, :], Device.Hip, reference_order=ref_order)[0]
        assert np.max(np.abs(y - want)) <= 1e-12
    assert np.array_equal(signal.sosfilt(sos, x, Device.Hip)[:16],
                          orc.sosfilt_f64(sos, x)[:16])


def test_signal_fixtures_and_edges():
    x = np.load(GOLD / "resample_x.npy")
    for name in ["butter", "cheby", "bessel", "notch"]:
        sos = np.load(GOLD / f"sos_{name}.npy")
        assert np.array_equal(signal.sosfilt(sos, x, Device.Hip),
                              np.load(GOLD / f"sosfilt_{name}.npy"))
    sos = np.load(GOLD / "sos_butter.npy")
    assert np.array_equal(signal.filtfilt(sos, x, Device.Hip), np.load(GOLD / "filtfilt_butter.npy"))
    # no sections: the input passes through; empty inputs
    xr = np.random.default_rng(0).standard_normal((3, 500))
    assert np.array_equal(signal.sosfilt_batched(np.zeros((0, 6)), xr, Device.Hip), xr)
    assert signal.sosfilt(sos, np.zeros(0), Device.Hip).shape == (0,)
    assert signal.sosfilt_batched(sos, np.zeros((0, 10)), Device.Hip).shape == (0, 10)


def test_device_tier_strided_inplace_unaligned():
    print("sosfilt device tier", flush=True)
    rng = np.random.default_rng(9)
    sos_np = _sos(3)
    sos = torch.tensor(sos_np, device="cuda:0")
    big = torch.tensor(rng.standard_normal((5, 3001)), device="cuda:0")
    x = big[:, :2999]                      # row stride 3001 (odd: scalar loads)
    ref = orc.sosfilt_f64(sos_np, x.cpu().numpy())
    y = device.sosfilt(x, sos)
    torch.cuda.synchronize()
    _check(y.cpu().numpy(), ref, True)
    # in place, aligned rows
    z = torch.tensor(rng.standard_normal((4, 4096)), device="cuda:0")
    zref = orc.filtfilt_f64(sos_np, z.cpu().numpy())
    device.sosfilt(z, sos, zero_phase=True, out=z)
    torch.cuda.synchronize()
    _check(z.cpu().numpy(), zref, False)
    zr = torch.tensor(rng.standard_normal((4, 4096)), device="cuda:0")
    zrref = orc.sosfilt_f64(sos_np, zr.cpu().numpy())
    device.sosfilt(zr, sos, reference_order=True, out=zr)
    torch.cuda.synchronize()
    assert np.array_equal(zr.cpu().numpy(), zrref)


def test_full_size_rows():
    # the benchmark shape: a sample of rows against the oracle
    print("sosfilt full size", flush=True)
    rows, n = 4096, 65536
    gen = torch.Generator(device="cuda:0").manual_seed(3)
    x = torch.randn((rows, n), generator=gen, dtype=torch.float64, device="cuda:0")
    sos_np = ss.butter(6, 0.15, output="sos")
    sos = torch.tensor(sos_np, device="cuda:0")
    y = device.sosfilt(x, sos)
    torch.cuda.synchronize()
    for r in (0, 1, 2047, 4095):
        ref = orc.sosfilt_f64(sos_np, x[r].cpu().numpy())
        _check(y[r].cpu().numpy()[None, :], ref[None, :], True)
    del x, y
    torch.cuda.empty_cache()


# Few rows run in chunks of 1024 or 2048 samples that a wave holds: one chunk
# and its edges, 64, 65 and 128 of each (a lane collects two states), the first
# row length beyond them, rows enough to take the longer chunks, odd pitches.
@pytest.mark.parametrize("S", [1, 2, 3, 4])
@pytest.mark.parametrize("rows,n", [(1, 1025), (3, 2048), (2, 2049), (1, 65536), (2, 65537),
                                    (1, 131072), (1, 131073), (2, 262144), (1, 262145),
                                    (40, 130001), (700, 6001), (4095, 1100)])
def test_register_chunks(S, rows, n):
    print(f"sosfilt register chunks S={S} rows={rows} n={n}", flush=True)
    x = np.random.default_rng(S + n).standard_normal((rows, n))
    sos = _sos(S, S + n)
    keep = sorted({0, rows // 2, rows - 1})
    want, zero = orc.sosfilt_f64(sos, x[keep]), orc.filtfilt_f64(sos, x[keep])
    sos_t = torch.tensor(sos, device="cuda")
    for pitch in (n, n + 1):
        buf = torch.zeros((rows, pitch), dtype=torch.float64, device="cuda")
        xt = buf[:, :n]
        xt.copy_(torch.tensor(x))
        out = torch.full((rows, pitch), np.nan, dtype=torch.float64, device="cuda")[:, :n]
        device.sosfilt(xt, sos_t, out=out)
        _check(out.cpu().numpy()[keep], want, True, sos, x[keep])
        device.sosfilt(xt, sos_t, zero_phase=True, out=out)
        _check(out.cpu().numpy()[keep], zero, False, sos, x[keep], zero_phase=True)
        device.sosfilt(xt, sos_t, zero_phase=True, out=xt)  # in place
        _check(xt.cpu().numpy()[keep], zero, False, sos, x[keep], zero_phase=True)


def test_register_chunks_unstable_and_nonfinite():
    """A growing filter whose transition powers overflow (2000 of them would,
    the row is shorter), and NaNs: finite exactly before the first."""
    r = np.random.default_rng(3)
    sos = np.array([[1.0, 0.2, 0.1, 1.0, -2 * 1.05 * np.cos(0.3), 1.05 ** 2]])
    x = r.standard_normal((3, 5000))
    print("sosfilt register chunks unstable", flush=True)
    y, ref = signal.sosfilt_batched(sos, x, Device.Hip), orc.sosfilt_f64(sos, x)
    assert np.all(np.isfinite(ref))
    # Compared where the reference loop is: the output grows 1e100 times over.
    run = np.maximum.accumulate(np.abs(ref), axis=1)
    assert np.max(np.abs(y - ref) / run) <= 1e-9
    x[1, 3000] = np.nan
    y = signal.sosfilt_batched(sos, x, Device.Hip)
    assert np.all(np.isfinite(y[1, :3000])) and np.all(np.isnan(y[1, 3000:]))
    assert np.all(np.isfinite(y[[0, 2]]))


def test_register_chunks_captured_with_small_scratch():
    """A capture whose stream's scratch holds the general path's states but
    not both directions': it is taken, and replays to the oracle's results."""
    n, sos = 131072, _sos(1, 5)
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((1, n), device="cuda", dtype=torch.float64, generator=g)
    sos_t, y = torch.tensor(sos, device="cuda"), torch.empty_like(x)
    print("sosfilt capture with small scratch", flush=True)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        device.sosfilt(x[:, :1025].contiguous(), sos_t, zero_phase=True)
        st.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            device.sosfilt(x, sos_t, zero_phase=True, out=y)
    for _ in range(3):
        x.copy_(torch.randn((1, n), device="cuda", dtype=torch.float64, generator=g))
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        xh = x.cpu().numpy()
        _check(y.cpu().numpy(), orc.filtfilt_f64(sos, xh), False, sos, xh, zero_phase=True)
