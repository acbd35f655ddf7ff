"""Performance cases of the filtering paths, as a user's program calls them.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call
(inputs, taps, a plan), ``run(state)`` is one pass through the public entry
points, ``work(case)`` the bytes and operations a pass cannot do without and
``exact(case, seed)`` the pass's outputs in 64 bits, by plain torch or numpy.

Sizes are those of the benchmark workloads, of the reference's own examples
and benchmarks, and of the tests.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from scir_amd import _lib, device, gpu
from scir_amd.ragged import RaggedPlan


def listed():
    return [
        # The reference's own FIR example: a batch small enough that launch
        # latency counts.
        dict(name="fir_small", kind="fir", rows=64, samples=16384, taps=31, precision="f32"),
        # The same call from host memory: the drop-in that a user of the
        # reference switches to first.
        dict(name="fir_host", kind="host", rows=64, samples=16384, taps=33),
        # A short filter over a large resident batch: a pass over memory.
        dict(name="fir_short", kind="fir", rows=4096, samples=65536, taps=33, precision="f32"),
        # A medium filter, the arithmetic left to the library, rows of odd
        # length (no row but the first is aligned).
        dict(name="fir_medium", kind="fir", rows=4096, samples=65535, taps=129, precision="auto"),
        # The headline: long band-pass filters over long rows with outliers.
        dict(name="fir_long", kind="fir", rows=2048, samples=262144, taps=512, precision="auto",
             outliers=0.01),
        # A long filter in the default precision of the device tier.
        dict(name="fir_long_f32", kind="fir", rows=1024, samples=65536, taps=1023,
             precision="f32"),
        # A filter longer than one transform block: FFT overlap-save.
        dict(name="fir_fft", kind="fir", rows=256, samples=262144, taps=16384, precision="fft32",
             outliers=0.01),
        # Signals of uneven length, each with its own filter (the default
        # precision of a plan): a quarter of the ragged benchmark batch.
        dict(name="ragged", kind="ragged", signals=2500, min_len=256, max_len=1 << 20, k_lo=15,
             k_hi=1023, layout=3, precision="f32"),
        # A training step of a filter: forward, gradient of the input and of
        # the taps.
        dict(name="vjp", kind="vjp", rows=1024, samples=65536, taps=255, precision="f32"),
        # The reference's resampling case (up 2, down 3, 31 taps), batched.
        dict(name="resample", kind="resample", rows=4096, samples=65536, up=2, down=3, taps=31),
        # The reference's sosfilt benchmark filter over a large batch.
        dict(name="sosfilt", kind="iir", rows=4096, samples=65536, order=6, cutoff=0.15,
             zero_phase=False),
        # Zero-phase filtering of a few long recordings (the reference's
        # filtfilt benchmark filter): too few rows to fill the device.
        dict(name="filtfilt", kind="iir", rows=32, samples=262144, order=4, cutoff=0.2,
             zero_phase=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _shape(rng, rows, samples, most):
    """Rows and samples spread over the logarithms of their ranges, at most
    `most` samples in all; half of the row lengths odd."""
    while True:
        b, n = _log_int(rng, *rows), _log_int(rng, *samples)
        if b * n <= most:
            return b, n | rng.randrange(2)


def draw(rng):
    kind = rng.choice(["fir", "fir", "fir", "fir", "host", "ragged", "vjp", "resample", "iir"])
    if kind == "fir":
        precision = rng.choice(["f32", "f32", "auto", "auto", "f32_exact", "fft32"])
        if precision == "fft32":
            b, n = _shape(rng, (1, 2048), (4096, 262144), 1 << 26)
            return dict(kind=kind, rows=b, samples=n, taps=_log_int(rng, 128, 16384),
                        precision=precision)
        while True:
            b, n = _shape(rng, (1, 4096), (256, 262144), 1 << 27)
            k = _log_int(rng, 1, 2048)
            if b * n * k <= 1 << 37:
                return dict(kind=kind, rows=b, samples=n, taps=k, precision=precision,
                            outliers=rng.choice([0.0, 0.01]))
    if kind == "host":
        b, n = _shape(rng, (1, 256), (256, 65536), 1 << 22)
        return dict(kind=kind, rows=b, samples=n, taps=_log_int(rng, 3, 513))
    if kind == "ragged":
        lo = _log_int(rng, 64, 4096)
        return dict(kind=kind, signals=_log_int(rng, 16, 1500), min_len=lo,
                    max_len=lo * _log_int(rng, 2, 256), k_lo=_log_int(rng, 3, 63),
                    k_hi=_log_int(rng, 64, 1023), layout=rng.randrange(1 << 30),
                    precision=rng.choice(["f32", "auto"]))
    if kind == "vjp":
        b, n = _shape(rng, (1, 1024), (1024, 65536), 1 << 25)
        return dict(kind=kind, rows=b, samples=n, taps=_log_int(rng, 3, 1023),
                    precision=rng.choice(["f32", "auto"]))
    if kind == "resample":
        up, down = rng.choice([(2, 3), (2, 3), (3, 2), (1, 2), (2, 1), (4, 3)])
        b, n = _shape(rng, (1, 4096), (256, 65536), 1 << 26)
        k = 31 if (up, down) == (2, 3) else 20 * max(up, down) + 1
        return dict(kind=kind, rows=b, samples=n, up=up, down=down, taps=k)
    b, n = _shape(rng, (1, 4096), (1024, 262144), 1 << 26)
    return dict(kind=kind, rows=b, samples=n, order=rng.choice([2, 4, 6, 8]),
                cutoff=round(rng.uniform(0.05, 0.4), 3), zero_phase=rng.random() < 0.5)


# ---- inputs -----------------------------------------------------------------


def _generator(seed, stream, where="cuda"):
    g = torch.Generator(device=where)
    g.manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _rows(shape, seed, stream, dtype=torch.float32, outliers=0.0):
    """N(0, 1) samples on the GPU, a share of them scaled by 1000."""
    g = _generator(seed, stream)
    x = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    if outliers:
        x *= torch.where(torch.rand(shape, generator=g, device="cuda") < outliers, 1000.0, 1.0)
    return x


def _sinc_filter(taps, lo, hi, beta=None):
    """Windowed-sinc band filter in float64: Hamming window, or Kaiser."""
    m = np.arange(taps) - (taps - 1) / 2
    w = np.kaiser(taps, beta) if beta else np.hamming(taps) if taps > 1 else np.ones(1)
    h = (hi * np.sinc(hi * m) - (lo * np.sinc(lo * m) if lo else 0.0)) * w
    f = 0.0 if not lo else (lo + hi) / 2
    return h / np.sum(h * np.cos(math.pi * m * f))


def _fir_taps(case, seed):
    """A low-pass, or for the long filters a band-pass; the band edges move
    a little with the seed."""
    shift = 0.002 * (int(seed) % 17)
    if case["taps"] >= 256:
        return _sinc_filter(case["taps"], 0.1 + shift, 0.3 + shift, 8.0).astype(np.float32)
    return _sinc_filter(case["taps"], 0.0, 0.2 + shift).astype(np.float32)


def _ragged_layout(case):
    rng = np.random.default_rng(case["layout"])
    n = case["signals"]
    lens = np.exp(rng.uniform(math.log(case["min_len"]), math.log(case["max_len"]), n))
    lens = np.round(lens).astype(np.int64)
    ks = rng.integers(case["k_lo"], case["k_hi"] + 1, n).astype(np.int64)
    offs = np.concatenate(([0], np.cumsum(lens)))
    b_offs = np.concatenate(([0], np.cumsum(ks)))
    return offs, b_offs


def _ragged_taps(case, seed):
    _, b_offs = _ragged_layout(case)
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, 5])
    cut = rng.uniform(0.05, 0.45, case["signals"])
    return np.concatenate([_sinc_filter(int(k), 0.0, c)
                           for k, c in zip(np.diff(b_offs), cut)]).astype(np.float32)


def _resample_taps(case):
    return case["up"] * _sinc_filter(case["taps"], 0.0, 1.0 / max(case["up"], case["down"]))


def _resample_len(case):
    off = (case["taps"] - 1) // 2
    conv = case["samples"] * case["up"] + case["taps"] - 1
    return max(0, -(-(conv - 2 * off) // case["down"]))


def _butterworth(case, seed):
    """Sections of a Butterworth low-pass of even order (bilinear transform)."""
    n = case["order"]
    k = math.tan(math.pi * (case["cutoff"] + 0.0005 * (int(seed) % 13)) / 2)
    sos = []
    for i in range(n // 2):
        q = 2 * math.sin(math.pi * (2 * i + 1) / (2 * n))
        a0 = 1 + q * k + k * k
        sos.append([k * k / a0, 2 * k * k / a0, k * k / a0, 1.0, 2 * (k * k - 1) / a0,
                    (1 - q * k + k * k) / a0])
    return np.array(sos)


# ---- the cases ----------------------------------------------------------------


def prepare(case, seed):
    kind, s = case["kind"], dict(case)
    if kind == "host":
        s["x"] = np.random.default_rng([int(seed) & 0x7FFFFFFF, 1]).standard_normal(
            (case["rows"], case["samples"]), dtype=np.float32)
        s["b"] = np.ascontiguousarray(_fir_taps(case, seed)[::-1])
        return s
    if kind == "ragged":
        offs, b_offs = _ragged_layout(case)
        s["plan"] = RaggedPlan(offs, b_offs, case["precision"])
        s["x"] = _rows((int(offs[-1]),), seed, 1)
        s["b"] = torch.tensor(_ragged_taps(case, seed), device="cuda")
        s["y"] = torch.empty_like(s["x"])
        return s
    shape = (case["rows"], case["samples"])
    wide = kind in ("resample", "iir")
    s["x"] = _rows(shape, seed, 1, torch.float64 if wide else torch.float32,
                   case.get("outliers", 0.0))
    if kind == "resample":
        s["h"] = torch.tensor(_resample_taps(case), device="cuda")
        s["y"] = torch.empty((case["rows"], _resample_len(case)), device="cuda",
                             dtype=torch.float64)
        return s
    if kind == "iir":
        s["sos"] = torch.tensor(_butterworth(case, seed), device="cuda")
        s["y"] = torch.empty_like(s["x"])
        return s
    s["b"] = torch.tensor(_fir_taps(case, seed), device="cuda")
    s["y"] = torch.empty_like(s["x"])
    if kind == "vjp":
        s["g"] = _rows(shape, seed, 2)
        s["dx"] = torch.empty_like(s["x"])
        s["db"] = torch.empty_like(s["b"])
    return s


def run(state):
    kind = state["kind"]
    if kind == "fir":
        return device.fir(state["x"], state["b"], state["precision"], out=state["y"])
    if kind == "host":
        return gpu.fir1d_batched_f32_auto(state["x"], state["b"], gpu.Device.Hip)
    if kind == "ragged":
        return state["plan"].execute(state["x"], state["b"], state["y"])
    if kind == "vjp":
        return (device.fir(state["x"], state["b"], state["precision"], out=state["y"]),
                device.vjp_dx(state["g"], state["b"], state["precision"], out=state["dx"]),
                device.vjp_db(state["g"], state["x"], state["taps"], out=state["db"]))
    if kind == "resample":
        x, h, y = state["x"], state["h"], state["y"]
        stream = torch.cuda.current_stream(x.device).cuda_stream
        p = ctypes.c_void_p
        _lib.check(_lib.lib().scir_hip_resample_poly_f64_dev(
            p(x.data_ptr()), x.stride(0), x.shape[0], x.shape[1], state["up"], state["down"],
            p(h.data_ptr()), h.numel(), p(y.data_ptr()), y.stride(0), p(stream)))
        return y
    return device.sosfilt(state["x"], state["sos"], zero_phase=state["zero_phase"],
                          out=state["y"])


def work(case):
    kind = case["kind"]
    if kind == "ragged":
        offs, b_offs = _ragged_layout(case)
        lens, ks = np.diff(offs), np.diff(b_offs)
        return dict(bytes=8 * int(offs[-1]) + 4 * int(b_offs[-1]),
                    flops=2 * int(np.sum(lens * ks)))
    n = case["rows"] * case["samples"]
    if kind == "resample":
        m = case["rows"] * _resample_len(case)
        return dict(bytes=8 * (n + m + case["taps"]),
                    flops=2 * m * -(-case["taps"] // case["up"]))
    if kind == "iir":
        # A section takes five multiplies and four adds a sample; a
        # zero-phase pass runs them twice.
        return dict(bytes=16 * n + 24 * case["order"],
                    flops=n * 9 * (case["order"] // 2) * (2 if case["zero_phase"] else 1))
    k = case["taps"]
    if kind == "vjp":
        # x, g in; y, dx, db out; three contractions.
        return dict(bytes=16 * n + 8 * k, flops=6 * k * n)
    if case.get("precision") == "fft32":
        # By transforms: the cheapest known way costs about 2.5 log2 of the
        # transform's length per real sample each way.
        return dict(bytes=8 * n + 4 * k, flops=int(5 * n * math.log2(4 * k)))
    return dict(bytes=8 * n + 4 * k, flops=2 * k * n)


# ---- the same in 64 bits --------------------------------------------------------


def _convolve(x, h, n_out):
    """Rows of x (float64) convolved with h, the first n_out samples."""
    size = 1 << (x.shape[-1] + h.shape[-1] - 1).bit_length()
    return torch.fft.irfft(torch.fft.rfft(x, size) * torch.fft.rfft(h, size), size)[..., :n_out]


def _by_rows(f, x, out_len, step=None):
    """f over groups of rows small enough for the transforms' scratch."""
    step = step or max(1, (1 << 25) // x.shape[1])
    out = torch.empty((x.shape[0], out_len), dtype=torch.float64, device=x.device)
    for r in range(0, x.shape[0], step):
        out[r:r + step] = f(x[r:r + step])
    return out


def _fir64(x, b):
    return _by_rows(lambda r: _convolve(r.double(), b, r.shape[1]), x, x.shape[1])


def _impulse_response(sos, n):
    """The cascade's first n outputs to a unit impulse."""
    v = np.zeros(n)
    v[0] = 1.0
    for b0, b1, b2, _, a1, a2 in sos:
        z1 = z2 = 0.0
        out = np.empty(n)
        for i in range(n):
            p = v[i]
            o = b0 * p + z1
            z1 = b1 * p - a1 * o + z2
            z2 = b2 * p - a2 * o
            out[i] = o
        v = out
    return v


def exact(case, seed):
    kind = case["kind"]
    if kind == "host":
        s = np.random.default_rng([int(seed) & 0x7FFFFFFF, 1]).standard_normal(
            (case["rows"], case["samples"]), dtype=np.float32)
        x = torch.tensor(s, device="cuda")
        b = torch.tensor(_fir_taps(case, seed), device="cuda").double()
        return _fir64(x, b).cpu().numpy()
    if kind == "ragged":
        offs, b_offs = _ragged_layout(case)
        x = _rows((int(offs[-1]),), seed, 1)
        b = torch.tensor(_ragged_taps(case, seed), device="cuda").double()
        y = torch.empty(x.shape, dtype=torch.float64, device="cuda")
        for i in range(case["signals"]):
            lo, hi = int(offs[i]), int(offs[i + 1])
            y[lo:hi] = _convolve(x[lo:hi].double(), b[int(b_offs[i]):int(b_offs[i + 1])], hi - lo)
        return y
    shape = (case["rows"], case["samples"])
    if kind == "resample":
        x = _rows(shape, seed, 1, torch.float64)
        h = _resample_taps(case)
        up, down, taps = case["up"], case["down"], case["taps"]
        m_out, off = _resample_len(case), (taps - 1) // 2
        pad = taps + down * up
        xp = torch.nn.functional.pad(x, (pad, pad + taps * up))
        y = torch.zeros((case["rows"], m_out), dtype=torch.float64, device="cuda")
        # Outputs m = up*j + r all read the taps k = n mod up, ... of one phase.
        for r in range(min(up, m_out)):
            first, count = off + down * r, -(-(m_out - r) // up)
            for k in range(first % up, taps, up):
                at = pad + (first - k) // up
                y[:, r::up] += h[k] * xp[:, at:at + down * (count - 1) + 1:down]
        return y
    if kind == "iir":
        # The filters settle in far fewer samples than the response kept.
        h = torch.tensor(_impulse_response(_butterworth(case, seed), 8192), device="cuda")
        x = _rows(shape, seed, 1, torch.float64)
        n = case["samples"]

        def both(r):
            y = _convolve(r, h, n)
            return _convolve(y.flip(-1), h, n).flip(-1) if case["zero_phase"] else y
        return _by_rows(both, x, n)
    x = _rows(shape, seed, 1, torch.float32, case.get("outliers", 0.0))
    b = torch.tensor(_fir_taps(case, seed), device="cuda").double()
    y = _fir64(x, b)
    if kind == "fir":
        return y
    g = _rows(shape, seed, 2)
    n, k = case["samples"], case["taps"]
    dx = _by_rows(lambda r: _convolve(r.double().flip(-1), b, n).flip(-1), g, n)
    size = 1 << (n + k - 1).bit_length()
    db = torch.zeros(k, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // n)
    for r in range(0, case["rows"], step):
        gf = torch.fft.rfft(g[r:r + step].double(), size)
        xf = torch.fft.rfft(x[r:r + step].double(), size)
        db += torch.fft.irfft((gf * xf.conj()).sum(0), size)[:k]
    return y, dx, db
