"""Chirp-z transforms in several passes against references: the five-pass form, batches and ragged classes
of three-pass ones, and more items than one launch takes.

Bars as in test_gpu_bluestein.py: FP64 relL2 1e-13, FP32 5e-7."""
import json

import numpy as np
import pytest

from conftest import rel_l2
from gfft_amd import api, inputs

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 1e-13, np.complex64: 5e-7}
VT = {np.complex128: api.COMPLEX_DOUBLE, np.complex64: api.COMPLEX_FLOAT}
BOTH = pytest.mark.parametrize("dtype", [np.complex128, np.complex64])


def fft(x):
    return np.fft.fft(x.astype(np.complex128), axis=-1)


def ifft(x):
    return np.fft.ifft(x.astype(np.complex128), axis=-1)


@BOTH
def test_five_passes(torch_cuda, tmp_path, monkeypatch, dtype):
    """A prime near 2^20 as a convolution of 2^21 = 128 * 128 * 128 points, named by a cache entry."""
    n = 1048573
    choice = [1 << 21, 128, 128, 128, 0, 16, 128, 32, 256, 16, 128, 32, 256, 16, 128]
    cache = tmp_path / "tune.json"
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(cache))
    for place in (api.OUT_OF_PLACE, api.IN_PLACE):
        api.Plan(n, VT[dtype], api.DFT, place).close()  # measured once, for the keys
    keys = list(json.loads(cache.read_text())["entries"])
    forced = tmp_path / "forced.json"
    forced.write_text('{"version": 2, "entries": {\n' + ",\n".join(f'"{k}": {choice}' for k in keys) + "\n}}\n")
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(forced))
    x = inputs.complex_normal(n, 3).astype(dtype)
    with api.Plan(n, VT[dtype], api.DFT, api.OUT_OF_PLACE) as pf, api.Plan(n, VT[dtype], api.IDFT, api.IN_PLACE) as pi:
        for p in (pf, pi):
            k = [q["kernel"] for q in json.loads(p.describe())["bluestein"]["passes"]]
            assert len(k) == 5 and k[0].endswith("chirp_in") and k[2].endswith("chirp_turn") and k[4].endswith("chirp_out"), k
        s = torch_cuda.from_numpy(x.copy()).cuda()
        o = torch_cuda.empty_like(s)
        pf.fft(s, o)
        pi.fft(s)
        torch_cuda.cuda.synchronize()
    assert rel_l2(o.cpu().numpy(), fft(x)) <= TOL[dtype]
    assert rel_l2(s.cpu().numpy(), ifft(x)) <= TOL[dtype]


@BOTH
@pytest.mark.parametrize("n", [4099, 11264, 65537])
def test_batches(torch_cuda, n, dtype):
    x = np.stack([inputs.complex_normal(n, 60 + b) for b in range(3)]).astype(dtype)
    kw = {"batch": 3, "flags": api.FLAG_NO_AUTOTUNE}
    with api.Plan(n, VT[dtype], api.DFT, api.OUT_OF_PLACE, **kw) as pf, api.Plan(n, VT[dtype], api.IDFT, api.IN_PLACE, **kw) as pi:
        assert len(json.loads(pf.describe())["bluestein"]["passes"]) == 3
        s = torch_cuda.from_numpy(x.copy()).cuda()
        o = torch_cuda.empty_like(s)
        pf.fft(s, o)
        pi.fft(s)
        torch_cuda.cuda.synchronize()
    for b in range(3):
        assert rel_l2(o.cpu().numpy()[b], fft(x[b])) <= TOL[dtype], b
        assert rel_l2(s.cpu().numpy()[b], ifft(x[b])) <= TOL[dtype], b


@BOTH
def test_ragged_classes(torch_cuda, dtype):
    lens = [11264, 4099, 512, 11264, 1009, 4099, 11264]
    x = inputs.complex_normal(sum(lens), 8).astype(dtype)
    for ttype, ref in ((api.DFT, fft), (api.IDFT, ifft)):
        p = api.RaggedPlan(lens, VT[dtype], ttype, flags=api.FLAG_NO_AUTOTUNE)
        d = torch_cuda.from_numpy(x.copy()).cuda()
        p.fft(d)
        torch_cuda.cuda.synchronize()
        y, off = d.cpu().numpy(), 0
        p.close()
        for i, n in enumerate(lens):
            assert rel_l2(y[off:off + n], ref(x[off:off + n])) <= TOL[dtype], i
            off += n


def test_more_items_than_a_launch_takes(torch_cuda):
    """65537 items: the passes run on 65535 of them and on 2.  Seven different ones, repeated."""
    torch = torch_cuda
    n, batch = 4099, 65537
    x = np.stack([inputs.complex_normal(n, 80 + b) for b in range(7)]).astype(np.complex64)
    d = torch.from_numpy(x).cuda().repeat((batch + 6) // 7, 1)[:batch].contiguous()
    with api.Plan(n, api.COMPLEX_FLOAT, api.DFT, api.IN_PLACE, batch=batch, flags=api.FLAG_NO_AUTOTUNE) as p:
        assert len(json.loads(p.describe())["bluestein"]["passes"]) == 3
        p.fft(d)
        torch.cuda.synchronize()
    first = d[:7].clone()
    for b in range(7):
        assert rel_l2(first[b].cpu().numpy(), fft(x[b])) <= TOL[np.complex64], b
    for lo in range(0, batch, 7 * 1024):
        part = torch.view_as_real(d[lo:lo + 7 * 1024])
        want = torch.view_as_real(first.repeat(1024, 1)[:part.shape[0]])
        assert torch.equal(part, want), lo
