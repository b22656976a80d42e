"""The transforms this library is timed on, through its Python binding (``gfft_amd.api``).

A case is one program's inner step: the plans exist, the arrays are in place, and one pass runs
the transforms on them.  Kinds:

  c2c     complex transforms of one length, ``batch`` of them back to back.  ``do`` is "fwd" or
          "inv" (out of place) or "pair" (forward, then inverse, in place: a filter's two
          transforms, which also leaves the values where they were)
  real    RDFT of 2n reals and the IRDFT back, out of place, in either packing
  ragged  complex transforms of many lengths in one buffer, forward then inverse in place
  host    complex transforms on arrays in host memory

Lengths are products of 2, 3, 5 and 7 or, on the chirp-z path, anything else.
"""
import math

import numpy as np
import torch

from gfft_amd import api, inputs

DEVICE = "cuda:0"


def listed():
    return [
        # one small transform per call, as a control loop or an interactive program issues them
        {"name": "single_1k_f64", "kind": "c2c", "n": 1024, "batch": 1, "prec": "f64", "do": "fwd"},
        # spectra of many short double-precision records, filtered in place
        {"name": "batch_1k_f64", "kind": "c2c", "n": 1024, "batch": 65536, "prec": "f64", "do": "pair"},
        # the same for single-precision records on the matrix cores (the flag a caller sets)
        {"name": "batch_4k_f32_mfma", "kind": "c2c", "n": 4096, "batch": 16384, "prec": "f32", "do": "fwd", "mfma": True},
        # short records whose length is a decimal number, as sample counts mostly are
        {"name": "batch_1000_f32", "kind": "c2c", "n": 1000, "batch": 16384, "prec": "f32", "do": "fwd"},
        # short records of a length with no small factors
        {"name": "batch_1009_f32", "kind": "c2c", "n": 1009, "batch": 8192, "prec": "f32", "do": "inv"},
        # one long record there and back: a convolution's two transforms
        {"name": "round_trip_16m_f32", "kind": "c2c", "n": 1 << 24, "batch": 1, "prec": "f32", "do": "pair"},
        # one long double-precision record of a decimal length
        {"name": "million_f64", "kind": "c2c", "n": 1000000, "batch": 1, "prec": "f64", "do": "fwd"},
        # one long record whose length is prime
        {"name": "prime_1m_f32", "kind": "c2c", "n": 1048573, "batch": 1, "prec": "f32", "do": "fwd"},
        # one long real signal, its n + 1 bins, and back
        {"name": "real_3m_f32", "kind": "real", "n": 3 << 19, "batch": 1, "prec": "f32", "bins": True},
        # frames of a real signal (2048 samples), spectra in GFFT's packing, and back
        {"name": "real_frames_f32", "kind": "real", "n": 1024, "batch": 8192, "prec": "f32", "bins": False},
        # records of uneven lengths in one buffer
        {"name": "ragged_4096_f32", "kind": "ragged", "count": 4096, "lo": 256, "hi": 65536, "prec": "f32", "lengths": 4096},
        # GFFT's own call: arrays in host memory
        {"name": "host_1m_f32", "kind": "host", "n": 1 << 20, "batch": 8, "prec": "f32"},
    ]


# ---------------------------------------------------------------------------------------
# drawn cases

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _is_smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _smooth(rng, lo, hi, step=1):
    """A product of 2, 3, 5 and 7 (a multiple of `step`) next to a log-uniform draw."""
    n = max(step, _log(rng, lo, hi) // step * step)
    while not _is_smooth(n):
        n += step
    return n


def _batch(rng, n, most):
    """How many transforms of length n: one in a third of the draws, else up to `most` points."""
    if rng.random() < 1 / 3 or 2 * n > most:
        return 1
    return max(1, _log(rng, max(2 * n, 1 << 12), most) // n)


def draw(rng):
    prec = rng.choice(["f32", "f64"])
    do = rng.choice(["fwd", "inv", "pair"])
    kind = rng.random()
    if kind < 0.40:
        n = _smooth(rng, 16, 1 << 22)
        return {"kind": "c2c", "n": n, "batch": _batch(rng, n, 1 << 24), "prec": prec, "do": do}
    if kind < 0.60:
        n = _log(rng, 11, 1 << 20)
        while _is_smooth(n):
            n += 1
        return {"kind": "c2c", "n": n, "batch": _batch(rng, n, 1 << 22), "prec": prec, "do": do}
    if kind < 0.75:
        n = _smooth(rng, 16, 1 << 22, 2)
        bins = rng.random() < 0.5
        return {"kind": "real", "n": n, "batch": 1 if bins else _batch(rng, n, 1 << 23), "prec": prec, "bins": bins}
    if kind < 0.87:
        hi = rng.choice([2048, 16384, 65536])
        return {"kind": "ragged", "count": _log(rng, 32, 4096), "lo": rng.choice([16, 256]), "hi": hi, "prec": prec,
                "lengths": rng.randrange(1, 100000)}
    if kind < 0.94:
        n = rng.choice([256, 4096])
        return {"kind": "c2c", "n": n, "batch": max(1, _log(rng, 1 << 12, 1 << 26) // n), "prec": "f32", "do": do, "mfma": True}
    n = _smooth(rng, 256, 1 << 21)
    return {"kind": "host", "n": n, "batch": _batch(rng, n, 1 << 22), "prec": prec}


# ---------------------------------------------------------------------------------------
# inputs and plans

def _types(c):
    if c["prec"] == "f64":
        return api.COMPLEX_DOUBLE, torch.complex128, torch.float64
    return api.COMPLEX_FLOAT, torch.complex64, torch.float32


def _lengths(c):
    return [int(v) for v in inputs.ragged_lengths(c["count"], c["lengths"], c["lo"], c["hi"])]


def _points(c):
    """Complex elements of the transforms' input."""
    return sum(_lengths(c)) if c["kind"] == "ragged" else c["n"] * c["batch"]


def _input(c, seed):
    """N(0, 1) samples: real ones for a real transform, numpy's for arrays in host memory."""
    _, ct, rt = _types(c)
    if c["kind"] == "host":
        r = np.random.default_rng(seed)
        x = r.standard_normal(2 * _points(c), dtype=np.float64 if c["prec"] == "f64" else np.float32)
        return x.view(np.complex128 if c["prec"] == "f64" else np.complex64).reshape(c["batch"], c["n"])
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    x = torch.randn(2 * _points(c), dtype=rt, device=DEVICE, generator=g)
    if c["kind"] == "real":
        return x.view(c["batch"], 2 * c["n"])
    x = torch.view_as_complex(x.view(-1, 2))
    return x if c["kind"] == "ragged" else x.view(c["batch"], c["n"])


def prepare(case, seed):
    c = case
    vt, ct, rt = _types(c)
    x = _input(c, seed)
    s = {"kind": c["kind"], "do": c.get("do"), "x": x}
    if c["kind"] == "ragged":
        lens = _lengths(c)
        s["fwd"] = api.RaggedPlan(lens, vt, api.DFT)
        s["inv"] = api.RaggedPlan(lens, vt, api.IDFT)
    elif c["kind"] == "real":
        flags = api.FLAG_R2C_BINS if c["bins"] else 0
        kw = {"flags": flags, "batch": c["batch"]}
        s["fwd"] = api.Plan(c["n"], vt, api.RDFT, api.OUT_OF_PLACE, **kw)
        s["inv"] = api.Plan(c["n"], vt, api.IRDFT, api.OUT_OF_PLACE, **kw)
        s["spectrum"] = torch.empty(c["batch"], c["n"] + (1 if c["bins"] else 0), dtype=ct, device=DEVICE)
        s["back"] = torch.empty_like(x)
    elif c["kind"] == "host":
        s["fwd"] = api.Plan(c["n"], vt, api.DFT, api.OUT_OF_PLACE, batch=c["batch"])
        s["out"] = np.empty_like(x)
    else:
        kw = {"flags": api.FLAG_SPLIT_MFMA if c.get("mfma") else 0, "batch": c["batch"]}
        place = api.IN_PLACE if c["do"] == "pair" else api.OUT_OF_PLACE
        if c["do"] != "inv":
            s["fwd"] = api.Plan(c["n"], vt, api.DFT, place, **kw)
        if c["do"] != "fwd":
            s["inv"] = api.Plan(c["n"], vt, api.IDFT, place, **kw)
        if c["do"] != "pair":
            s["out"] = torch.empty_like(x)
    return s


def run(state):
    s = state
    if s["kind"] == "real":
        s["fwd"].fft(s["x"], s["spectrum"])
        s["inv"].fft(s["spectrum"], s["back"])
        return {"spectrum": s["spectrum"], "back": s["back"]}
    if s["kind"] == "ragged" or s["do"] == "pair":
        s["fwd"].fft(s["x"])
        s["inv"].fft(s["x"])
        return {"x": s["x"]}
    s["inv" if s["do"] == "inv" else "fwd"].fft(s["x"], s["out"])
    return {"out": s["out"]}


def work(case):
    c = case
    eb = 16 if c["prec"] == "f64" else 8
    if c["kind"] == "ragged":
        lens = _lengths(c)
        return {"bytes": 2 * 2 * eb * sum(lens), "flops": 2 * sum(5 * n * math.log2(n) for n in lens)}
    n, b = c["n"], c["batch"]
    one = 2 * eb * n * b
    if c["kind"] == "real":
        # 2n reals: half the complex transform's operations, each way
        return {"bytes": 2 * one, "flops": 2 * 2.5 * 2 * n * math.log2(2 * n) * b}
    times = 2 if c.get("do") == "pair" else 1
    return {"bytes": times * one, "flops": times * 5 * n * math.log2(n) * b}


def exact(case, seed):
    """The same outputs in 64 bits."""
    c = case
    x = _input(c, seed)
    if c["kind"] == "real":
        x = x.double()
        X = torch.fft.rfft(x)
        if not c["bins"]:
            n = c["n"]
            packed = X[:, :n].clone()
            packed[:, 0] = torch.complex(X[:, 0].real, X[:, n].real)
            X = packed
        return {"spectrum": X, "back": x}
    if c["kind"] == "host":
        return {"out": np.fft.fft(x.astype(np.complex128))}
    x = x.to(torch.complex128)
    if c["kind"] == "ragged" or c["do"] == "pair":
        return {"x": x}
    return {"out": (torch.fft.ifft if c["do"] == "inv" else torch.fft.fft)(x)}
