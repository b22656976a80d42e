"""What the autotuner measures and reports."""
import json

import numpy as np
import pytest

from conftest import rel_l2
from gfft_amd import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mib,suffix", [(0, "|class|nt"), (256, "|class")])
def test_ragged_classes_tuned_with_the_stores_they_run_with(torch_cuda, tmp_path, monkeypatch, mib, suffix):
    """A class's last pass stores non-temporally where the whole batch is larger than the limit, not the
    class: its choice is measured and cached under that."""
    cache = tmp_path / "tune.json"
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(cache))
    monkeypatch.setenv("GFFTX_NT_STORE_MIB", str(mib))
    lens = [8192, 20000, 20000, 8192, 49152]
    x = inputs.complex_normal(sum(lens), 5)
    p = api.RaggedPlan(lens, api.COMPLEX_DOUBLE, api.DFT)
    d = torch_cuda.from_numpy(x.copy()).cuda()
    p.fft(d)
    torch_cuda.cuda.synchronize()
    y = d.cpu().numpy()
    p.close()
    off = 0
    for n in lens:
        assert rel_l2(y[off:off + n], np.fft.fft(x[off:off + n])) <= 1e-13
        off += n
    keys = [k for k in json.loads(cache.read_text())["entries"] if "|class" in k]
    assert len(keys) == 3 and all(k.endswith(suffix) for k in keys), keys
