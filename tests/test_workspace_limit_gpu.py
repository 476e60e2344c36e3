"""Calls whose preferred split of the solve does not fit a workspace limit take
fewer waves: in every entry point where it is the fixed workspace (the same bits),
in the server alone where it is its budget (the same fluxes but for the order of
the k-term sums: of at most 50 terms, which 1e-12 of the largest flux holds)."""
import re

import numpy as np
import pytest

from socrates_amd import runes as R
from socrates_amd import synth
from socrates_amd.serve import Server
from test_gpu_parity import NBAND
from test_zz_no_alloc import _device, _outs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()


def close(a, b):
    return np.abs(a - b).max() <= 1e-12 * np.abs(b).max()


def test_noalloc_near_its_limit():
    # 550 columns need 67.6 MB with 4 waves per column, of the 67.1 MB there are
    case = synth.make_case(550, 90, "lw", NBAND["lw"], seed=71, cloudy=True)
    arrs = _device(case)
    res = []
    for f in (R.runes, R.runes_noalloc):
        name, kw = R.case_call(case, "lw", device_arrays=arrs, out=_outs(case))
        res.append(f(kw.pop("n_profile"), kw.pop("n_layer"), name, kw.pop("i_source"), **kw))
    for k in ("flux_up", "flux_down"):
        assert np.array_equal(res[1][k].cpu().numpy(), res[0][k].cpu().numpy()), k


@pytest.mark.parametrize("src", ["sw", "lw"])
def test_serve_at_its_budget(src):
    case = synth.make_case(8, 60, src, NBAND[src], seed=72, cloudy=True)
    ref = R.runes_case(case, src)
    srv = Server(precision="fp64", hbm_budget_gb=1e-5, n_slots=1)
    try:
        with pytest.raises(R.SocgpuError) as e:
            srv.submit(*R.case_call(case, src))
    finally:
        srv.close()
    least = int(re.search(r"needs (\d+) bytes", str(e.value)).group(1))
    srv = Server(precision="fp64", hbm_budget_gb=(least + 1000) / 2.0 ** 30, n_slots=1)
    try:
        out = srv.wait(srv.submit(*R.case_call(case, src)))
    finally:
        srv.close()
    for k in ("flux_up", "flux_down"):
        assert close(np.asarray(out[k]), np.asarray(ref[k])), k
