"""The triple-column solve's split (clear layers four at a time above the call's
cloud top, a lane per region below it, 16 k-terms per wave) at the sizes where
it changes, against the oracle with the parity tests' tolerance (check_fp64:
flux within 1e-10 relative, 1e-9 W m-2 or 1e-11 of the column's largest, plus
the oracle's spread under one-ulp changes of its exponentials)."""
import numpy as np
import pytest

from oracle import oracle
from socrates_amd import runes as R
from socrates_amd import synth
from test_gpu_parity import NBAND, SPEC, check_fp64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()


def make(src, P, L, n_cloudy, seed):
    """A triple-column case whose lowest n_cloudy layers hold cloud of either
    type, both or none; one column without any."""
    case = synth.make_case(P, L, src, NBAND[src], seed=seed, cloudy=True, overlap="triple")
    rng = np.random.default_rng(seed + 1)
    st, cv = (rng.uniform(0.05, 0.45, (L, P)) * rng.integers(0, 2, (L, P)) for _ in range(2))
    st[L - n_cloudy:, 0] = 0.3
    if P > 2:
        st[:, 1] = cv[:, 1] = 0.0
    for f in (st, cv):
        f[:L - n_cloudy] = 0.0
    lwc = 1.0e-4 * np.exp(rng.normal(0.0, 1.0, (2, L, P))) / case.density
    case.cloud_frac, case.conv_frac = st, cv
    case.liq_mmr, case.liq_conv_mmr = lwc[0] * st, lwc[1] * cv
    return case


# (columns, layers, cloudy layers): 0 to 5 clear layers, a cloud top in the last
# layer, the fewest layers, the LDS classes' last and next, cloud throughout
SHAPES = [(1, 2, 2), (3, 2, 1), (3, 12, 11), (3, 12, 10), (3, 12, 9), (3, 12, 8), (3, 13, 8), (5, 17, 1), (3, 96, 40),
          (3, 97, 33), (3, 144, 144), (3, 145, 20), (2, 192, 60)]


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_sizes_match_oracle(src, shape):
    P, L, n_cloudy = shape
    case = make(src, P, L, n_cloudy, 6000 + 10 * L + n_cloudy + (src == "sw"))
    ref = oracle.runes(case, SPEC[src], None)
    sp = {k: np.zeros_like(ref[k]) for k in ("flux_up", "flux_down", "flux_direct")}
    for _ in range(2):
        j = oracle.runes(case, SPEC[src], None, variant="jitter")
        for k in sp:
            sp[k] = np.maximum(sp[k], np.abs(j[k] - ref[k]))
    check_fp64(R.runes_case(case, src, precision="fp64"), ref, "triple %s %s" % (src, shape), src,
               case.layer_heat_capacity, spread=sp)
