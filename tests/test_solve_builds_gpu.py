"""Builds of the column solve that test_solve_rows_gpu does not reach: few layers (up
to 24, four lanes per solve) at the edges of their split, and the builds for aerosols
and for the general gas optics (GA9 files) on both sides of every line between builds
(24, 96 and 144 layers) with shallow and deep cloud; and the triple column's mixed
form at the sizes where its split changes.

Tolerances: the parity tests' (check_fp64: 1e-10 relative, 1e-9 W m-2 or 1e-11 of the
column's largest; check_mixed), in FP64 plus twice the oracle's own largest movement
in the column under one-ulp changes of its exponentials (exp_spread of
test_aerosol_gpu). Columns with cloud up to their top are compared in FP64 only: the
mixed form's heating-rate bound is that of cloud in the troposphere."""
import numpy as np
import pytest

import test_solve_rows_gpu
import test_tri_rows_gpu
from oracle import oracle
from socrates_amd import runes as R
from socrates_amd import synth
from test_aerosol_gpu import exp_spread, files_of
from test_ga9_gpu import MCICA_GA9, NAME, SPEC_GA9, WM
from test_gpu_parity import check_fp64, check_mixed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def spectra():
    R.register_default_spectra()
    for src in ("sw", "lw"):
        R.set_spectrum(NAME[src], SPEC_GA9[src])
    R.set_mcica(MCICA_GA9, sw_spectrum_name=NAME["sw"], lw_spectrum_name=NAME["lw"])


def compare(case, name, files, src, label, mixed):
    ref = oracle.runes(case, files[src], files["mcica"] if case.l_cloud else None)
    check_fp64(R.runes_case(case, name, precision="fp64"), ref, label, src, case.layer_heat_capacity,
               spread=exp_spread(case, files, src), factor=2.0)
    if mixed:
        check_mixed(R.runes_case(case, name, precision="mixed"), ref, label + " mixed")


# (columns, layers, cloudy layers): one layer, a full lane and one over; the two-solve
# cloudy part full (8) and one over; cloud from the top; the most layers and one over;
# no cloud; a group of several rounds
@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", [(1, 3, 2), (3, 4, 3), (3, 5, 2), (3, 8, 8), (3, 9, 9), (5, 20, 8), (5, 20, 9),
                                   (3, 23, 12), (3, 24, 24), (3, 25, 25), (2, 24, 0), (40, 24, 6)])
def test_few_layers(src, shape):
    P, L, n = shape
    case = test_solve_rows_gpu.make(src, P, L, n, 8000 + 10 * L + n + (src == "sw"))
    compare(case, src, files_of("synth"), src, "few %s %s" % (src, shape), n < L)


SHAPES = [(3, 10, 5), (3, 24, 10), (3, 25, 10), (3, 60, 33), (3, 96, 20), (3, 97, 40), (3, 144, 30), (3, 145, 40)]


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", SHAPES)
def test_aerosols(src, shape):
    P, L, n = shape
    case = test_solve_rows_gpu.make(src, P, L, n, 8500 + 10 * L + n + (src == "sw"))
    synth.add_aerosols(case, 2, 8600 + L)
    compare(case, src, files_of("synth"), src, "aerosol %s %s" % (src, shape), True)


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", SHAPES)
def test_general_optics(src, shape):
    P, L, n = shape
    case = test_solve_rows_gpu.make(src, P, L, n, 8700 + 10 * L + n + (src == "sw"))
    case.wm_mix_ratio = WM.copy()
    compare(case, NAME[src], files_of("x_ga9_x"), src, "ga9 %s %s" % (src, shape), True)


@pytest.mark.parametrize("src", ["lw", "sw"])
@pytest.mark.parametrize("shape", [s for s in test_tri_rows_gpu.SHAPES if s[2] < s[1]])
def test_triple_mixed(src, shape):
    P, L, n = shape
    case = test_tri_rows_gpu.make(src, P, L, n, 6000 + 10 * L + n + (src == "sw"))
    ref = oracle.runes(case, files_of("synth")[src], None)
    check_mixed(R.runes_case(case, src, precision="mixed"), ref, "triple mixed %s %s" % (src, shape))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("L", [20, 97, 145])
def test_waves_per_block(L, precision):
    """Blocks of 1, 2 and 4 waves (more LDS than 64 KB above 96 layers) give the same bits."""
    case = synth.add_aerosols(test_solve_rows_gpu.make("sw", 7, L, L // 3, 8900 + L), 2, 8901)
    saved = R.get_tile(precision)
    try:
        out = []
        for waves in (1, 2, 4):
            R.set_tile(precision, 0, waves)
            out.append(R.runes_case(case, "sw", precision=precision))
    finally:
        R.set_tile(precision, saved["recompute"], saved["waves_per_block"], saved["waves_per_simd"])
    for o in out[1:]:
        for k in o:
            assert np.array_equal(o[k], out[0][k]), k
