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


@pytest.mark.parametrize("n,ttype", [(3628800, api.DFT), (3628800, api.IRDFT), (65537, api.DFT)])
def test_describe_lists_the_fastest_candidates(torch_cuda, tmp_path, monkeypatch, n, ttype):
    """Dozens of candidates: describe() has room for its list, and no two of them read alike."""
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setenv("GFFTX_TUNE_CANDIDATES", "20")
    with api.Plan(n, api.COMPLEX_FLOAT, ttype, api.OUT_OF_PLACE) as p:
        d = json.loads(p.describe())
    splits, ms = [t["split"] for t in d["tuned"]], [t["ms"] for t in d["tuned"]]
    assert 2 <= len(splits) <= 32 and ms == sorted(ms)
    assert len(set(splits)) == len(splits)
    if n == 65537:
        m = [int(s.split(":")[0]) for s in splits]
        assert all(v >= 2 * n - 1 for v in m) and all(s.count("x") == 2 and s.count("/") == 3 for s in splits)


def test_cache_entries_that_are_no_split(torch_cuda, tmp_path, monkeypatch):
    """A cache file may hold anything: lengths that do not multiply to n are not run."""
    cache = tmp_path / "tune.json"
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(cache))
    n, lens = 1 << 17, [20000, 49152]

    def run():
        x = inputs.complex_normal(n, 6)
        with api.Plan(n, api.COMPLEX_DOUBLE, api.DFT, api.IN_PLACE) as p:
            d = torch_cuda.from_numpy(x.copy()).cuda()
            p.fft(d)
            assert rel_l2(d.cpu().numpy(), np.fft.fft(x)) <= 1e-13
        x = inputs.complex_normal(sum(lens), 7)
        p = api.RaggedPlan(lens, api.COMPLEX_DOUBLE, api.DFT)
        d = torch_cuda.from_numpy(x.copy()).cuda()
        p.fft(d)
        y = d.cpu().numpy()
        p.close()
        assert rel_l2(y[:lens[0]], np.fft.fft(x[:lens[0]])) <= 1e-13
        assert rel_l2(y[lens[0]:], np.fft.fft(x[lens[0]:])) <= 1e-13

    run()  # measured, for the keys
    keys = list(json.loads(cache.read_text())["entries"])
    assert len(keys) == 3
    forged = tmp_path / "forged.json"
    forged.write_text('{"version": 2, "entries": {\n' + ",\n".join(f'"{k}": [256, 128]' for k in keys) + "\n}}\n")
    monkeypatch.setenv("GFFTX_TUNE_CACHE", str(forged))
    run()
