"""Performance cases of the STFT engine: the requests its users make, through
the public entry points of ``occastft_amd``.

A case is a dict of plain values: the entry point (``kind``), the sizes and
the option string.

  device   Runner.run_device          one signal resident on the GPU
  strided  Runner.run_strided_device  many equal signals resident on the GPU
  batch    Runner.run_batch_device    many uneven requests resident on the GPU
  host     Runner.stft                the reference's ActivateSTFT: numpy in, numpy out

Ranges: windows 2^6 .. 2^20, 2^14 .. 2^27 samples per signal, overlap 0 .. 0.9
(fractions that give odd hops among them), every output layout, every window
function, with and without DC removal, FP32 and the matrix-core form.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import occastft_amd as ostft

DEVICE = "cuda:0"

# window functions: option -> (cosine coefficients, samples of the period less N)
_COS = {
    "--hanning_window": ((0.5, -0.5), -1),
    "--hamming_window": ((0.54, -0.46), -1),
    "--blackman_window": ((0.42, -0.5, 0.08), 0),
    "--nuttall_window": ((0.355768, -0.487396, 0.144232, -0.012604), 0),
    "--blackman_harris_window": ((0.35875, -0.48829, 0.14128, -0.01168), 0),
    "--flattop_window": ((0.21557895, -0.41663158, 0.277263158, -0.083578947, 0.006947368), 0),
}
_LAYOUTS = ("", "--half_complex_return", "--magnitude_return", "--power_return", "--half_spectrum_return")


def listed() -> list[dict]:
    return [
        # a short clip, the shortest request of the serving mix: launch latency is all of it
        dict(name="clip_256", kind="device", samples=1 << 14, exp=8, overlap=0.75,
             options="--hamming_window --power_return"),
        # the reference's own call on a signal in host memory, copies included
        dict(name="activate_1024", kind="host", samples=1 << 20, exp=10, overlap=0.5,
             options="--hanning_window --remove_dc"),
        # a long recording with the smallest, a middle and a large one-kernel
        # window, in the two layouts the reference's runners return
        dict(name="record_64", kind="device", samples=100_000_000, exp=6, overlap=0.5,
             options="--hanning_window --remove_dc"),
        dict(name="record_512_complex", kind="device", samples=100_000_000, exp=9, overlap=0.0,
             options="--hanning_window --remove_dc --half_complex_return"),
        dict(name="record_4096", kind="device", samples=100_000_000, exp=12, overlap=0.5,
             options="--hanning_window --remove_dc"),
        # a recording whose length, overlap and hop divide nothing; odd exponents
        # from 13 on return the reference's penultimate stage
        dict(name="ragged_8192", kind="device", samples=30_000_019, exp=13, overlap=0.45,
             options="--blackman_harris_window --magnitude_return"),
        # large windows, for fine frequency resolution: dense spectrograms at
        # both ends of the range, and a plain block transform in between
        dict(name="large_65536", kind="device", samples=1 << 27, exp=16, overlap=0.75,
             options="--blackman_window --remove_dc --power_return"),
        dict(name="large_262144", kind="device", samples=1 << 27, exp=18, overlap=0.0,
             options="--blackman_window --remove_dc"),
        dict(name="large_1048576", kind="device", samples=1 << 27, exp=20, overlap=0.75,
             options="--blackman_window --remove_dc --power_return"),
        # thousands of equal signals (channels, clips of a data set) at once
        dict(name="signals_256", kind="strided", count=4096, samples=1 << 18, exp=8, overlap=0.5,
             options="--hanning_window --half_spectrum_return"),
        # the same on the matrix cores
        dict(name="signals_1024_fp16", kind="strided", count=1024, samples=1 << 18, exp=10, overlap=0.5,
             options="--hanning_window --half_spectrum_return --mfma_fp16"),
        # a serving batch: uneven lengths, windows, overlaps and window functions
        dict(name="mixed_batch", kind="batch", count=256, trace=5, shortest=1 << 14, longest=1 << 22,
             exp_low=8, exp_high=13, options="--power_return"),
    ]


def _log_int(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _options(rng, exp: int, matrix: bool) -> str:
    opts = [rng.choice([*_COS, "--hanning_window", "--blackman_window", ""]), rng.choice(_LAYOUTS)]
    if rng.random() < 0.5:
        opts.append("--remove_dc")
    if matrix:
        opts.append("--mfma_fp16")
    return " ".join(o for o in opts if o)


def draw(rng) -> dict:
    kind = rng.choices(["device", "strided", "batch", "host"], [12, 3, 2, 2])[0]
    if kind == "batch":
        low = rng.randint(6, 11)
        return dict(kind="batch", count=_log_int(rng, 16, 256), trace=rng.randrange(1 << 20), shortest=1 << 14,
                    longest=1 << rng.randint(18, 22), exp_low=low, exp_high=rng.randint(low, 13),
                    options=rng.choice(_LAYOUTS))
    exp = rng.randint(6, 20) if kind == "device" else rng.randint(6, 13)
    overlap = rng.choice([0.0, 0.25, 0.5, 0.5, 0.75, 0.75, round(rng.uniform(0.0, 0.9), 2)])
    matrix = kind == "strided" and exp in (6, 8, 10) and rng.random() < 0.5
    case = dict(kind=kind, exp=exp, overlap=overlap, options=_options(rng, exp, matrix))
    # the samples that the listed cases' largest output and work allow
    most = {"device": (1 << 27) * min(1.0, 4.0 * (1.0 - overlap)), "host": 1 << 22,
            "strided": (1 << 28) * (1.0 - overlap)}[kind]
    if kind == "strided":
        case["samples"] = _log_int(rng, 1 << 14, 1 << 20)
        case["count"] = max(2, int(_log_int(rng, 1 << 20, int(most)) / case["samples"]))
    else:
        case["samples"] = _log_int(rng, 1 << max(14, exp), int(most))
    return case


# ------------------------------------------------------------ geometry, in the reference's float32

def _geometry(samples: int, exp: int, overlap: float) -> tuple[int, int]:
    """-> (frames, hop)"""
    f = np.float32
    n, step = f(1 << exp), f(1) - f(overlap)
    q = f(samples) / n + f(1) if overlap == 0.0 else f(samples) / (n * step) + f(1)
    return int(np.trunc(np.float64(q))), int(n * step)


def _out_floats(frames: int, exp: int, options: str) -> int:
    n = 1 << exp
    if "--power_return" in options:
        return frames * (n // 2 + 1)
    if "--half_spectrum_return" in options:
        return frames * (n + 2)
    return frames * n


def _requests(case: dict) -> list[dict]:
    """The requests of a batch: one list for a case, whatever its inputs hold."""
    rng = np.random.default_rng(case["trace"])
    out = []
    for _ in range(case["count"]):
        out.append(dict(
            samples=int(round(math.exp(rng.uniform(math.log(case["shortest"]), math.log(case["longest"]))))),
            exp=int(rng.integers(case["exp_low"], case["exp_high"] + 1)),
            overlap=float(rng.choice([0.0, 0.25, 0.5, 0.75])),
            options=" ".join([str(rng.choice(["--hanning_window", "--hamming_window", "--blackman_window"])),
                              case["options"]])))
    return out


def _batch_layout(case: dict):
    """-> [(request, input offset, output offset, output floats)], input floats, output floats"""
    at_in = at_out = 0
    rows = []
    for r in _requests(case):
        frames, _ = _geometry(r["samples"], r["exp"], r["overlap"])
        n = _out_floats(frames, r["exp"], r["options"])
        rows.append((r, at_in, at_out, n))
        at_in += (r["samples"] + 3) // 4 * 4
        at_out += (n + 3) // 4 * 4
    return rows, at_in, at_out


# ------------------------------------------------------------ inputs

def _signal(n: int, seed: int) -> torch.Tensor:
    """Five tones and noise on a small offset, as a recording holds: n floats on the GPU."""
    rng = np.random.default_rng(seed)
    tones = [(rng.uniform(0, 0.5), rng.uniform(0.1, 1.0), rng.uniform(0, 2 * np.pi)) for _ in range(5)]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    x = torch.randn(n, device=DEVICE, generator=gen).mul_(0.05).add_(0.1)
    for s in range(0, n, 1 << 25):
        part = x[s: s + (1 << 25)]
        k = torch.arange(s, s + part.numel(), dtype=torch.float64, device=DEVICE)
        for f, a, ph in tones:
            # whole turns come off in float64, the sine itself is float32
            part += (2 * np.pi * torch.frac(k * f + ph / (2 * np.pi))).float().sin_().mul_(a)
    return x


_RUNNER = None


def _runner() -> "ostft.Runner":
    """The engine handle: a program makes one and keeps it."""
    global _RUNNER
    if _RUNNER is None:
        _RUNNER = ostft.Runner(0)
    return _RUNNER


def prepare(case: dict, seed: int) -> dict:
    state = dict(kind=case["kind"], runner=_runner())
    if case["kind"] == "host":
        state["x"] = _signal(case["samples"], seed).cpu().numpy()
        state["call"] = (case["exp"], case["overlap"], case["options"])
        return state
    if case["kind"] == "batch":
        rows, n_in, n_out = _batch_layout(case)
        x = _signal(n_in, seed)
        state["out"] = torch.zeros(n_out, device=DEVICE)
        state["jobs"] = [(x[i: i + r["samples"]], ostft.parse_options(r["options"], r["exp"], r["overlap"]),
                          state["out"][o: o + n]) for r, i, o, n in rows]
        return state
    state["params"] = ostft.parse_options(case["options"], case["exp"], case["overlap"])
    frames, _ = _geometry(case["samples"], case["exp"], case["overlap"])
    n = _out_floats(frames, case["exp"], case["options"])
    if case["kind"] == "strided":
        state["x"] = _signal(case["count"] * case["samples"], seed).view(case["count"], case["samples"])
        state["out"] = torch.zeros(case["count"], (n + 3) // 4 * 4, device=DEVICE)
    else:
        state["x"] = _signal(case["samples"], seed)
        state["out"] = torch.zeros(n, device=DEVICE)
    return state


def run(state: dict):
    r = state["runner"]
    if state["kind"] == "device":
        return r.run_device(state["x"], state["params"], out=state["out"])
    if state["kind"] == "strided":
        return r.run_strided_device(state["x"], state["params"], out=state["out"])
    if state["kind"] == "batch":
        r.run_batch_device(state["jobs"])
        return state["out"]
    return r.stft(state["x"], *state["call"])


# ------------------------------------------------------------ what a pass cannot do without

def _work(samples: int, exp: int, overlap: float, options: str) -> tuple[float, float]:
    n = 1 << exp
    frames, hop = _geometry(samples, exp, overlap)
    floats = _out_floats(frames, exp, options)
    # the reference's complex layout returns the first half of the frames' spectra
    done = (frames + 1) // 2 if "--half_complex_return" in options else frames
    span = min(samples, (done - 1) * hop + n)
    return 4.0 * (span + floats), done * (2.5 * n * exp + 3.0 * n)


def work(case: dict) -> dict:
    if case["kind"] == "batch":
        parts = [_work(r["samples"], r["exp"], r["overlap"], r["options"]) for r in _requests(case)]
    else:
        parts = [_work(case["samples"], case["exp"], case["overlap"], case["options"])] * case.get("count", 1)
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ------------------------------------------------------------ the same in float64, in plain torch

def _window64(options: str, n: int):
    for name, (coef, less) in _COS.items():
        if name in options.split():
            k = torch.arange(n, dtype=torch.float64, device=DEVICE) * (2 * math.pi / (n + less))
            return sum(c * torch.cos(j * k) for j, c in enumerate(coef))
    return None


def _stft64(x: torch.Tensor, exp: int, overlap: float, options: str, out: torch.Tensor) -> None:
    """The layout's float64 values of signal x into the flat tensor `out`."""
    n = 1 << exp
    frames, hop = _geometry(x.numel(), exp, overlap)
    win = _window64(options, n)
    power, spectrum = "--power_return" in options, "--half_spectrum_return" in options
    complex_, magnitude = "--half_complex_return" in options, "--magnitude_return" in options
    per = _out_floats(1, exp, options) * (2 if complex_ else 1)  # floats a frame fills
    if complex_:
        frames = (frames + 1) // 2
    stage = exp >= 13 and exp % 2 == 1 and not (power or spectrum)  # the reference stops one stage early
    chunk = max(1, (1 << 25) // n)
    x = torch.nn.functional.pad(x, (0, max(0, (frames - 1) * hop + n - x.numel())))
    for f0 in range(0, frames, chunk):
        f1 = min(frames, f0 + chunk)
        y = x[f0 * hop: (f1 - 1) * hop + n].double().unfold(0, n, hop)
        y = y * win if win is not None else y.clone()
        if "--remove_dc" in options.split():
            y -= y.mean(dim=1, keepdim=True)
        if stage:
            y = torch.cat([torch.fft.fft(y[:, 0::2].contiguous()), torch.fft.fft(y[:, 1::2].contiguous())], dim=1)
        elif power or spectrum:
            y = torch.fft.rfft(y)
        else:
            y = torch.fft.fft(y)
        if power:
            y = y.real.square() + y.imag.square()
        elif spectrum or complex_:
            y = torch.view_as_real(y)
        else:
            y = y.abs() if magnitude else math.sqrt(2.0) * y.real.abs()
        y = y.reshape(-1)[: out.numel() - f0 * per]
        out[f0 * per: f0 * per + y.numel()] = y


def exact(case: dict, seed: int):
    if case["kind"] == "batch":
        rows, n_in, n_out = _batch_layout(case)
        x = _signal(n_in, seed)
        out = torch.zeros(n_out, dtype=torch.float64, device=DEVICE)
        for r, i, o, n in rows:
            _stft64(x[i: i + r["samples"]], r["exp"], r["overlap"], r["options"], out[o: o + n])
        return out
    frames, _ = _geometry(case["samples"], case["exp"], case["overlap"])
    n, count = _out_floats(frames, case["exp"], case["options"]), case.get("count", 1)
    x = _signal(count * case["samples"], seed).view(count, case["samples"])
    out = torch.zeros(count, n, dtype=torch.float64, device=DEVICE)
    for y in range(count):
        _stft64(x[y], case["exp"], case["overlap"], case["options"], out[y])
    if case["kind"] == "strided":
        return out
    return out[0].cpu().numpy() if case["kind"] == "host" else out[0]
