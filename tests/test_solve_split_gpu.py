"""A call's k-term sums are grouped alike wherever it is made: alone, in a batch, in the
fixed workspace, and in the server whatever its budget, where a wave that takes all of
a column's groups in turn has the bits of a wave for each."""
import re

import numpy as np
import pytest

from socrates_amd import runes as R
from socrates_amd import synth
from socrates_amd.serve import Server
from test_ga9_gpu import MCICA_GA9, NAME, SPEC_GA9, WM
from test_gpu_parity import NBAND
from test_zz_no_alloc import _device, _outs

pytestmark = pytest.mark.gpu

FLUXES = ("flux_up", "flux_down", "flux_direct", "heating_rate")


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()


def served(case, src, precision, budget_gb):
    srv = Server(precision=precision, hbm_budget_gb=budget_gb, n_slots=1)
    try:
        return srv.wait(srv.submit(*R.case_call(case, src)))
    finally:
        srv.close()


def least_gb(case, src, precision):
    srv = Server(precision=precision, hbm_budget_gb=1e-6, n_slots=1)
    try:
        with pytest.raises(R.SocgpuError) as e:
            srv.submit(*R.case_call(case, src))
    finally:
        srv.close()
    return (int(re.search(r"needs (\d+) bytes", str(e.value)).group(1)) + 8) / 2.0 ** 30


# 550 x 90 infra-red: fits the fixed workspace with fewer groups than a call of its
# size takes otherwise; 8 columns: a group per round; 40: three rounds a group
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("src,P,L,kind", [("lw", 550, 90, "cloud"), ("sw", 8, 60, "cloud"), ("lw", 8, 100, "cloud"),
                                          ("sw", 40, 60, "cloud"), ("lw", 8, 50, "clear"), ("sw", 8, 70, "aerosol"),
                                          ("lw", 17, 150, "aerosol"), ("lw", 8, 20, "cloud"),
                                          ("sw", 40, 10, "cloud")])
def test_server_has_the_bits_of_the_call_alone(src, P, L, kind, precision):
    case = synth.make_case(P, L, src, NBAND[src], seed=P + L, cloudy=kind != "clear")
    if kind == "aerosol":
        synth.add_aerosols(case, 2, P + L)
    ref = R.runes_case(case, src, precision=precision)
    for budget in (16.0, least_gb(case, src, precision)):
        out = served(case, src, precision, budget)
        for k in FLUXES:
            assert np.array_equal(np.asarray(out[k]), np.asarray(ref[k])), (k, budget)


def test_batch_and_fixed_workspace_have_the_bits_of_the_call_alone():
    case = synth.make_case(560, 90, "lw", NBAND["lw"], seed=73, cloudy=True)
    arrs = _device(case)
    res = []
    for f in (R.runes, R.runes_noalloc):
        name, kw = R.case_call(case, "lw", device_arrays=arrs, out=_outs(case))
        res.append(f(kw.pop("n_profile"), kw.pop("n_layer"), name, kw.pop("i_source"), **kw))
    res.append(R.runes_batch([R.case_call(case, "lw", device_arrays=arrs, out=_outs(case))])[0])
    for k in FLUXES:
        if k in res[0]:
            for r in res[1:]:
                assert np.array_equal(r[k].cpu().numpy(), res[0][k].cpu().numpy()), k


@pytest.mark.parametrize("src", ["sw", "lw"])
def test_server_general_optics(src):
    for s in ("sw", "lw"):
        R.set_spectrum(NAME[s], SPEC_GA9[s])
    R.set_mcica(MCICA_GA9, sw_spectrum_name=NAME["sw"], lw_spectrum_name=NAME["lw"])
    for P, L in ((20, 60), (9, 100), (20, 20)):
        case = synth.make_case(P, L, src, NBAND[src], seed=P + L, cloudy=True)
        case.wm_mix_ratio = WM.copy()
        ref = R.runes_case(case, NAME[src], precision="mixed")
        out = served(case, NAME[src], "mixed", least_gb(case, NAME[src], "mixed"))
        for k in FLUXES:
            assert np.array_equal(np.asarray(out[k]), np.asarray(ref[k])), (k, P, L)
