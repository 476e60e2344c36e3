"""The triple-column solve's workspace rows for numbers of k-terms that no file of the
package has: 21 of a wave's 64 lanes' worth and one over, three full waves (63), and
64, the one number whose rows are not padded to lines, because padded ones would need
more room than callers' workspaces have held. Against the oracle with the tolerance of
test_tri_rows_gpu."""
import os
import re
import sys

import numpy as np
import pytest
import torch

import test_tri_rows_gpu
from oracle import oracle
from socrates_amd import runes as R
from test_gpu_parity import SPEC, check_fp64, check_mixed
from test_zz_no_alloc import FIELDS, _outs

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import make_spectra  # noqa: E402

pytestmark = pytest.mark.gpu


def spectrum(path, n_g):
    """sp_lw_synth with n_g major k-terms, spread evenly over its bands."""
    n = len(make_spectra.LW_BANDS)
    bands = [(gas, n_g // n + (b < n_g % n), minor) for b, (gas, _, minor) in enumerate(make_spectra.LW_BANDS)]
    text = open(SPEC["lw"]).read()
    block = "\n".join(make_spectra.block5(np.random.default_rng(n_g), bands, {1: 1, 2: 2, 3: 3}))
    new, found = re.subn(r"\*BLOCK: TYPE =    5:.*?\*END[^\n]*", lambda m: block, text, flags=re.S)
    assert found == 1
    path.write_text(new)
    return str(path)


@pytest.mark.parametrize("n_g", [21, 22, 63, 64, 65])
def test_rows_by_number_of_terms(tmp_path, n_g):
    f = spectrum(tmp_path / "sp", n_g)
    name = "lw_%d_terms" % n_g
    R.set_spectrum(name, f)
    case = test_tri_rows_gpu.make("lw", 5, 30, 17, 7000 + n_g)
    ref = oracle.runes(case, f, None)
    sp = {k: np.zeros_like(ref[k]) for k in ("flux_up", "flux_down", "flux_direct")}
    for _ in range(2):
        j = oracle.runes(case, f, None, variant="jitter")
        for k in sp:
            sp[k] = np.maximum(sp[k], np.abs(j[k] - ref[k]))
    check_fp64(R.runes_case(case, name, precision="fp64"), ref, "triple %d terms" % n_g, "lw",
               case.layer_heat_capacity, spread=sp)
    check_mixed(R.runes_case(case, name, precision="mixed"), ref, "triple %d terms mixed" % n_g)


def test_room_of_a_call(tmp_path):
    """A 64-term call needs no more room in the fixed workspace than with a lane per
    k-term and three regions of 4 words: records of 21 words per layer and its level
    temperature, scalars, band and cloud records, overlaps, level sums, the solve's
    state, 52 words of alignment and 1280 bytes of descriptor."""
    P, L, NB = 400, 90, 9
    name = "lw_64_terms"
    R.set_spectrum(name, spectrum(tmp_path / "sp", 64))
    case = test_tri_rows_gpu.make("lw", P, L, 17, 7100)
    arrs = {k: torch.from_numpy(np.ascontiguousarray(getattr(case, k))).cuda()
            for k in FIELDS + ("conv_frac", "liq_conv_mmr", "liq_conv_dim")}
    arrs["cos_zenith_angle"] = torch.from_numpy(np.ascontiguousarray(case.cos_zen)).cuda()
    _, kw = R.case_call(case, name, device_arrays=arrs, out=_outs(case))
    with pytest.raises(R.SocgpuError) as e:
        R.runes_noalloc(kw.pop("n_profile"), kw.pop("n_layer"), name, kw.pop("i_source"), **kw)
    need = int(re.search(r"needs (\d+) bytes", str(e.value)).group(1))
    words = (P * L * 21 + P * (L + 1) + P * 7 + P * NB * L * 4 + P * NB * 4 + 2 + P * NB * L * 8 + P * (L + 1) * 18 +
             P * (L + 1) * 3 + P * L * 3 * 4 * 64)
    assert need <= 1280 + 8 * (words + 52)
