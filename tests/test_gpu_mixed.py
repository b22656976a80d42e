"""Run-time mixed-radix tiles on the GPU against the long-double oracle: lengths of one butterfly,
of two to five stages, with idle threads, at the largest sizes a tile takes; single passes, first
and later passes, real transforms and offset tables (ragged classes).  The bars are the library's
own: FP64 1e-13, FP32 2e-7 relative L2."""
import json

import numpy as np
import pytest

from conftest import rel_l2
from gfft_amd import api, inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 1e-13, np.complex64: 2e-7}
VT = {np.complex128: api.COMPLEX_DOUBLE, np.complex64: api.COMPLEX_FLOAT}


def host(t):
    import torch

    torch.cuda.synchronize()
    return t.cpu().numpy()


def kernels(p):
    return [k["kernel"] for k in json.loads(p.describe())["passes"]]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,batch", [(3, 5), (6, 300), (9, 57), (10, 1), (12, 65), (15, 257), (18, 129), (35, 9), (63, 4),
                                     (100, 21), (243, 3), (625, 2), (1000, 7), (1215, 1), (2401, 3), (4000, 2), (6561, 1),
                                     (7938, 2), (8100, 1), (15876, 2), (16200, 1)])
def test_single_pass(torch_cuda, dtype, n, batch):
    if dtype == np.complex128 and n > 8192:
        pytest.skip("FP64 tiles take up to 8192 points")
    x = np.stack([inputs.complex_normal(n, 10 * n + b) for b in range(batch)]).astype(dtype)
    fwd = np.stack([O.ref_fft(r, 1) for r in x])
    inv = np.stack([O.ref_fft(r, -1) for r in x]) / n
    print(f"case mixed n={n} batch={batch} dtype={np.dtype(dtype).name}", flush=True)
    with api.Plan(n, VT[dtype], api.DFT, api.OUT_OF_PLACE, batch=batch, flags=api.FLAG_NO_AUTOTUNE) as p:
        # 15876 = 14*14*9*9 and 16200 = 15*15*9*8 would take more than 1024 threads: passes
        assert n > 15000 or (len(kernels(p)) == 1 and kernels(p)[0].startswith("mixed_"))
        s = torch_cuda.from_numpy(x).cuda()
        o = torch_cuda.full_like(s, float("nan"))
        p.fft(s, o)
        assert rel_l2(host(o), fwd) <= TOL[dtype]
        assert np.array_equal(host(s), x)
    with api.Plan(n, VT[dtype], api.IDFT, api.IN_PLACE, batch=batch, flags=api.FLAG_NO_AUTOTUNE) as p:
        d = torch_cuda.from_numpy(x).cuda()
        p.fft(d)
        assert rel_l2(host(d), inv) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("passes,batch", [("18,20", 3), ("1000,30", 1), ("100,243", 2), ("2048,27", 1), ("1215,64", 1),
                                          ("36,35,50", 1), ("256,512", 2), ("1920,21", 1)])
def test_passes(torch_cuda, monkeypatch, dtype, passes, batch):
    """First (T->E) and later (T->T) passes, rows cut off at the end of the sequences included."""
    monkeypatch.setenv("GFFTX_PASSES", passes)
    n = int(np.prod([int(v) for v in passes.split(",")]))
    monkeypatch.setenv("GFFTX_AUTOTUNE", "0")
    x = np.stack([inputs.complex_normal(n, 3 * n + b) for b in range(batch)]).astype(dtype)
    print(f"case mixed passes={passes} batch={batch} dtype={np.dtype(dtype).name}", flush=True)
    for tt, sign, scale in ((api.DFT, 1, 1.0), (api.IDFT, -1, 1.0 / n)):
        ref = np.stack([O.ref_fft(r, sign) for r in x]) * scale
        with api.Plan(n, VT[dtype], tt, api.OUT_OF_PLACE, batch=batch) as p:
            if any(k.startswith("mixed_") and "truefalse" in k for k in kernels(p)):
                assert len(kernels(p)) == passes.count(",") + 1
            s = torch_cuda.from_numpy(x).cuda()
            o = torch_cuda.full_like(s, float("nan"))
            p.fft(s, o)
            assert rel_l2(host(o), ref) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,batch,bins", [(6, 9, False), (10, 1, True), (18, 33, False), (50, 1, True), (1000, 3, False),
                                          (1250, 1, True), (2430, 2, False), (8000, 1, True)])
def test_real_single_pass(torch_cuda, dtype, n, batch, bins):
    """RDFT with the split after the last stage, IRDFT with the pre-split before the first one."""
    z = inputs.complex_normal(n * batch, 77 + n).astype(dtype).reshape(batch, n)
    rt = np.float64 if dtype == np.complex128 else np.float32
    ref = np.fft.rfft(z.view(rt).astype(np.float64), axis=-1)
    if not bins:
        ref = np.concatenate([ref[:, :1].real + 1j * ref[:, n:].real, ref[:, 1:n]], axis=1)
    flags = api.FLAG_NO_AUTOTUNE | (api.FLAG_R2C_BINS if bins else 0)
    print(f"case mixed real n={n} batch={batch} bins={bins} dtype={np.dtype(dtype).name}", flush=True)
    with api.Plan(n, VT[dtype], api.RDFT, api.OUT_OF_PLACE, batch=batch, flags=flags) as pf, \
            api.Plan(n, VT[dtype], api.IRDFT, api.OUT_OF_PLACE, batch=batch, flags=flags) as pi:
        assert kernels(pf)[0].endswith("e_split") and kernels(pi)[0].endswith("e_presplit")
        s = torch_cuda.from_numpy(z).cuda()
        o = torch_cuda.full((batch, ref.shape[1]), float("nan"), dtype=s.dtype, device="cuda")
        pf.fft(s, o)
        assert rel_l2(host(o), ref) <= TOL[dtype]
        back = torch_cuda.full_like(s, float("nan"))
        pi.fft(o, back)
        assert rel_l2(host(back), z) <= 2 * TOL[dtype]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_ragged_classes(torch_cuda, dtype):
    """Lengths without a compiled tile, reached through a ragged batch's offset table."""
    lengths = [1000, 63, 1000, 2430, 100, 63, 12500, 1000, 6000, 100]
    x = inputs.complex_normal(sum(lengths), 5).astype(dtype)
    p = api.RaggedPlan(lengths, VT[dtype], api.DFT, flags=api.FLAG_NO_AUTOTUNE)
    d = torch_cuda.from_numpy(x).cuda()
    p.fft(d)
    y = host(d)
    off = 0
    for n in lengths:
        assert rel_l2(y[off:off + n], O.ref_fft(x[off:off + n], 1)) <= TOL[dtype], n
        off += n
    p.close()
