"""The column solve's layer split (16 lanes per solve, 6, 9 or 12 layers per
lane by build; the cloudy layers of a column in LDS up to 32 of them, in
private memory above) at the sizes where it changes, against the oracle with
the parity tests' tolerance: flux within 1e-10 relative, 1e-9 W m-2 or 1e-11 of
the column's largest, plus the reference's own movement under one-ulp changes
of its exponentials (check_fp64, oracle_spread)."""
import numpy as np
import pytest

from oracle import oracle
from socrates_amd import runes as R
from socrates_amd import synth
from test_gpu_parity import MCICA, NBAND, SPEC, check_fp64, check_mixed, oracle_spread

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()


def make(src, P, L, n_cloudy, seed):
    """A McICA case whose lowest n_cloudy layers hold cloud: overcast,
    partial and clear ones, every layer of the first column; one column
    without any, one overcast throughout."""
    case = synth.make_case(P, L, src, NBAND[src], seed=seed, cloudy=True)
    rng = np.random.default_rng(seed + 1)
    frac = rng.uniform(0.05, 1.0, (L, P)) * rng.integers(0, 2, (L, P))
    frac[:, 0] = rng.uniform(0.3, 0.9, L)
    if P > 2:
        frac[:, 1] = 0.0
        frac[:, 2] = 1.0
    frac[:L - n_cloudy] = 0.0
    lwc = 1.0e-4 * np.exp(rng.normal(0.0, 1.0, (L, P)))
    case.cloud_frac, case.liq_mmr = frac, lwc / case.density * frac
    return case


# (columns, layers, cloudy layers): one layer per lane and less; 16 lanes full
# and one over; the two-solve cloudy part full (32) and one over; the builds'
# last and next sizes; cloud from the top layer; no cloud at all; more columns
# than the one-round split takes
SHAPES = [(3, 2, 1), (3, 15, 4), (3, 16, 16), (3, 17, 8), (3, 60, 32), (3, 60, 33), (3, 96, 96), (3, 97, 9),
          (3, 144, 40), (3, 145, 33), (3, 192, 192), (4, 50, 0), (18, 33, 7)]


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_sizes_match_oracle(src, shape):
    P, L, n_cloudy = shape
    case = make(src, P, L, n_cloudy, 4000 + 10 * L + n_cloudy + (src == "sw"))
    ref = oracle.runes(case, SPEC[src], MCICA)
    check_fp64(R.runes_case(case, src, precision="fp64"), ref, "%s %s" % (src, shape), src,
               case.layer_heat_capacity, spread=oracle_spread(case, src, True))
    # the mixed form's absolute bounds are those of cloud in the troposphere: the
    # thin top layers with cloud in them heat by 1e4 K/day
    if n_cloudy < L:
        check_mixed(R.runes_case(case, src, precision="mixed"), ref, "mixed %s %s" % (src, shape))
