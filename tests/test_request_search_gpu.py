"""Batches whose number of calls lies around the steps of the kernels' search for
an item's call (64 and 4096 starts a round), with calls that take no part in some
kernels: each call's results are those it has alone, bit for bit. Layer counts
around the output kernel's tiles (15 layers)."""
import numpy as np
import pytest

from socrates_amd import runes as R
from socrates_amd import synth
from test_gpu_parity import NBAND

pytestmark = pytest.mark.gpu
FIELDS = ("flux_up", "flux_down", "flux_direct", "heating_rate")


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()


@pytest.mark.parametrize("n", [2, 64, 65, 129, 4097])
def test_batch_sizes(n):
    kinds = [("lw", 1, 15, {}), ("sw", 2, 16, dict(cloudy=True)), ("lw", 3, 14, dict(cloudy=True, overlap="triple")),
             ("sw", 17, 31, {}), ("lw", 1, 98, dict(cloudy=True)), ("sw", 1, 30, {})]
    cases = [(s, synth.make_case(P, L, s, NBAND[s], seed=80 + i, **kw)) for i, (s, P, L, kw) in enumerate(kinds)]
    alone = [R.runes_case(c, s) for s, c in cases]
    pick = np.random.default_rng(n).integers(0, len(cases), n)
    outs = R.runes_batch([R.case_call(cases[k][1], cases[k][0]) for k in pick])
    for k, o in zip(pick, outs):
        for f in FIELDS:
            assert np.array_equal(np.asarray(o[f]), np.asarray(alone[k][f])), (n, kinds[k], f)
        fl = {f: np.asarray(o[f]) for f in FIELDS}
        net = fl["flux_down"] - fl["flux_up"]
        c = cases[k][1]
        # the heating is the divergence of the fluxes given out: one subtraction more
        got = fl["heating_rate"] * c.layer_heat_capacity
        assert np.abs(got - (net[:-1] - net[1:])).max() <= 1e-12 * np.abs(fl["flux_down"]).max()
