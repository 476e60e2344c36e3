"""Every build of the kernel-level two-stream solve against the oracle: the splits
for few layers (up to 3 layers in one lane, up to 12 in four groups of 3), and the
mixed form of the builds of 3, 6, 9 and 12 layers per group with blocks of 32 and
of 64 columns.

Tolerances. FP64: those of test_two_stream_gpu (1e-10 relative, 1e-9 W m-2 or 1e-11
of the column's scale). The infra-red inputs are absorbing layers no thinner than
0.01, where a last-bit change of an exponential moves 1 - T - R (1.7e-3 at least) by
1.3e-13 of itself and so the quadratic source by 1e-11 of a Planck term of at most
some tens of W m-2. Mixed: its stated bound of 0.05 W m-2."""
import numpy as np
import pytest

from socrates_amd import runes as R
from socrates_amd import synth
from test_two_stream_gpu import _check, _oracle_terms

pytestmark = pytest.mark.gpu


def make(P, L, G, isolir, flags=(1, 1)):
    """n_layer 1 as the top layer of a two-layer case."""
    c = synth.make_two_stream_case(P, max(L, 2), isolir, seed=900 + 7 * L + isolir, n_term=G, omc_range=(-1.0, 0.0),
                                   tau_range=(-2.0, 2.0), l_scale_solar=flags[0], l_ir_source_quad=flags[1])
    if L == 1:
        c["n_layer"] = 1
        for k in ("tau", "omega", "asymmetry"):
            c[k] = np.ascontiguousarray(c[k][:, :1])
        for k in ("diff_planck", "diff_planck_2", "adjust_solar_ke"):
            c[k] = np.ascontiguousarray(c[k][:1])
    return c


@pytest.mark.parametrize("isolir", [1, 2])
@pytest.mark.parametrize("flags", [(1, 1), (0, 0)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (13, 1, 5), (65, 2, 1), (64, 3, 2), (5, 4, 13), (64, 5, 1), (13, 11, 5),
                                   (9, 12, 8), (9, 13, 8)])
def test_few_layers(shape, flags, isolir):
    P, L, G = shape
    tsc = make(P, L, G, isolir, flags)
    ref = _oracle_terms(tsc)
    gpu = R.two_stream_case(tsc, "fp64")
    _check(gpu, ref, None, "fp64 isolir=%d %s" % (isolir, shape))
    if isolir == 1:
        assert np.abs(np.asarray(gpu["flux_direct"]) - ref[2]).max() <= 1e-10 * np.abs(ref[2]).max()


# 8193 solves are the fewest that blocks of 64 columns take
@pytest.mark.parametrize("isolir", [1, 2])
@pytest.mark.parametrize("P,G", [(13, 5), (2731, 3)])
@pytest.mark.parametrize("L", [3, 12, 13, 48, 49, 96, 97, 144, 145, 192])
def test_mixed_builds(L, P, G, isolir):
    tsc = make(P, L, G, isolir)
    ref = _oracle_terms(tsc)
    gpu = R.two_stream_case(tsc, "mixed")
    for k, r in zip(("flux_up", "flux_down", "flux_direct"), ref):
        if k != "flux_direct" or isolir == 1:
            assert np.abs(np.asarray(gpu[k]) - r).max() <= 0.05, k
