"""The band kernel's split (16 lanes per column, 6, 9 or 12 layers per lane by
build, 4 columns per block, the bands over the block's waves) at the sizes where
it changes, against the oracle with the parity tests' tolerance (check_fp64: flux
within 1e-10 relative, 1e-9 W m-2 or 1e-11 of the column's largest, plus the
oracle's spread under one-ulp changes of its exponentials)."""
import numpy as np
import pytest

from oracle import oracle
from ga9_cases import MCICA_GA9, SPEC_GA9
from socrates_amd import runes as R
from socrates_amd import synth
from test_gpu_parity import NBAND, SPEC, check_fp64, oracle_spread

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()
    for s in ("sw", "lw"):
        R.set_spectrum("%s_ga9" % s, SPEC_GA9[s])
    R.set_mcica(MCICA_GA9, sw_spectrum_name="sw_ga9", lw_spectrum_name="lw_ga9")


# columns: a block with 1, 3 and 4, one over, and more blocks than take the most
# waves; layers around 16, the builds' last and next
@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", [(1, 2), (3, 15), (4, 16), (5, 17), (5, 96), (3, 97), (3, 144), (2, 145), (2, 192),
                                   (2060, 5)])
def test_clear_sky_matches_oracle(src, shape):
    P, L = shape
    case = synth.make_case(P, L, src, NBAND[src], seed=5200 + L + (src == "sw"))
    ref = oracle.runes(case, SPEC[src], None)
    check_fp64(R.runes_case(case, src, precision="fp64"), ref, "%s %s" % (src, shape), src,
               case.layer_heat_capacity, spread=oracle_spread(case, src, False))


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", [(5, 17), (3, 97), (2, 145)])
def test_general_gas_optics_match_oracle(src, shape):
    P, L = shape
    case = synth.make_case(P, L, src, NBAND[src], seed=5300 + L + (src == "sw"))
    case.wm_mix_ratio = np.array([4.7255e-7, 9.637e-7, 0.23139, 0.0, 0.0, 2.0e-10, 3.0e-10, 0.0, 1.0e-10, 0.0])
    ref = oracle.runes(case, SPEC_GA9[src], None)
    sp = {k: np.zeros_like(ref[k]) for k in ("flux_up", "flux_down", "flux_direct")}
    for _ in range(2):
        j = oracle.runes(case, SPEC_GA9[src], None, variant="jitter")
        for k in sp:
            sp[k] = np.maximum(sp[k], np.abs(j[k] - ref[k]))
    check_fp64(R.runes_case(case, src + "_ga9", precision="fp64"), ref, "ga9 %s %s" % (src, shape), src,
               case.layer_heat_capacity, spread=sp)
