"""Stores of the passes that carry a real transform's split: through the L2 or not, the bits are the
same, and both match numpy's real FFT.  Bars: FP64 relL2 1e-13, FP32 5e-7 (twice that for a round trip)."""
import json

import numpy as np
import pytest

from conftest import rel_l2
from gfft_amd import api, inputs

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-13, "f32": 5e-7}

# last passes with half rows of 256, 128 and 64 bytes at 2 MiB and more (forward); first passes at
# 12 MiB and more (inverse, FP32)
CASES = [
    (3 << 19, "f32", "256,96,64"), (1 << 18, "f32", "1024,256"), (1 << 21, "f32", "128,128,128"),
    (1 << 17, "f64", "1024,128"), (1 << 19, "f64", "256,128,16"), (1 << 20, "f64", "256,64,64"),
]


@pytest.mark.parametrize("n,prec,passes", CASES)
def test_split_passes(torch_cuda, monkeypatch, n, prec, passes):
    torch = torch_cuda
    vt, rt, ct = (api.DOUBLE, np.float64, np.complex128) if prec == "f64" else (api.FLOAT, np.float32, np.complex64)
    x = inputs.complex_normal(n, 17).astype(ct).view(rt)
    X = np.fft.rfft(x.astype(np.float64))
    ref = np.concatenate([[X[0].real + 1j * X[n].real], X[1:n]])
    monkeypatch.setenv("GFFTX_PASSES", passes)
    out = {}
    for on in (1, 0):
        monkeypatch.setenv("GFFTX_THROUGH_STORE", str(on))
        with api.Plan(n, vt, api.RDFT, api.OUT_OF_PLACE) as pf, api.Plan(n, vt, api.IRDFT, api.OUT_OF_PLACE) as pi:
            assert json.loads(pf.describe())["passes"][-1]["kernel"].endswith("_split")
            assert json.loads(pi.describe())["passes"][0]["kernel"].endswith("_presplit")
            s = torch.from_numpy(x.view(ct)).cuda()
            o, b = torch.empty_like(s), torch.empty_like(s)
            pf.fft(s, o)
            pi.fft(o, b)
            torch.cuda.synchronize()
            out[on] = o.cpu().numpy(), b.cpu().numpy()
    for got, want in zip(out[1], out[0]):
        assert np.array_equal(got, want)
    assert rel_l2(out[1][0], ref) <= TOL[prec]
    assert rel_l2(out[1][1], x.view(ct)) <= 2 * TOL[prec]
