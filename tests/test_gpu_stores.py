"""Store kinds of multi-pass plans: written through the L2 or not, the bits are the same."""
import numpy as np
import pytest

from gfft_amd import api, inputs

pytestmark = pytest.mark.gpu

# around the 2 MiB where it begins, whole and partial 128-byte rows, two to five passes
CASES = [
    ("c2c", 1 << 18, 1, "f32"), ("c2c", (1 << 18) - (1 << 8), 1, "f32"), ("c2c", 1 << 17, 1, "f64"),
    ("c2c", 1000000, 1, "f64"), ("c2c", 44100, 20, "f32"), ("c2c", 1 << 22, 1, "f32"),
    ("c2c", 300007, 1, "f32"), ("c2c", 150001, 3, "f64"),
    ("real", 3 << 19, 1, "f32"), ("real", 1 << 18, 2, "f64"),
]


@pytest.mark.parametrize("kind,n,batch,prec", CASES)
def test_write_through_stores_change_no_result(torch_cuda, monkeypatch, kind, n, batch, prec):
    torch = torch_cuda
    vt, ct = (api.COMPLEX_DOUBLE, np.complex128) if prec == "f64" else (api.COMPLEX_FLOAT, np.complex64)
    x = torch.from_numpy(inputs.complex_normal(n * batch, 91).astype(ct)).cuda()
    flags = api.FLAG_NO_AUTOTUNE

    def run(on):
        monkeypatch.setenv("GFFTX_THROUGH_STORE", str(on))
        outs = []
        kinds = (api.DFT, api.IDFT) if kind == "c2c" else (api.RDFT, api.IRDFT)
        src = x
        for t in kinds:
            with api.Plan(n, vt, t, api.OUT_OF_PLACE, batch=batch, flags=flags) as p:
                dst = torch.empty_like(x)
                p.fft(src, dst)
                torch.cuda.synchronize()
                outs.append(dst.cpu().numpy())
                src = dst
        return outs

    for a, b in zip(run(1), run(0)):
        assert np.array_equal(a, b)
        assert np.isfinite(a.view(a.real.dtype)).all()
