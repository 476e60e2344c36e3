"""The kernel-level two-stream solve's split of a column over 16 waves (3, 6, 9
or 12 layers each by build) at the sizes where it changes, with solve counts
that do not fill the last wave, against the oracle with the tolerance of
test_two_stream_gpu (1e-10 relative, 1e-9 W m-2 or 1e-11 of the column's scale,
plus the oracle's own spread in the infra-red)."""
import numpy as np
import pytest

from socrates_amd import runes as R
from socrates_amd import synth
from test_two_stream_gpu import _check, _oracle_terms, _spread

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("isolir", [1, 2])
@pytest.mark.parametrize("shape", [(1, 2, 1), (13, 16, 7), (64, 17, 1), (13, 48, 5), (13, 49, 5), (3, 96, 3),
                                   (3, 97, 22), (5, 144, 2), (5, 145, 2), (7, 192, 3)])
def test_split_sizes_match_oracle(isolir, shape):
    P, L, G = shape
    tsc = synth.make_two_stream_case(P, L, isolir, seed=70 + L + isolir, n_term=G, omc_range=(-3.0, 0.0))
    ref = _oracle_terms(tsc)
    gpu = R.two_stream_case(tsc, "fp64")
    _check(gpu, ref, _spread(tsc, ref) if isolir == 2 else None, "fp64 isolir=%d %s" % (isolir, shape))
    if isolir == 1:
        assert np.abs(np.asarray(gpu["flux_direct"]) - ref[2]).max() <= 1e-10 * np.abs(ref[2]).max()


@pytest.mark.parametrize("isolir", [1, 2])
@pytest.mark.parametrize("shape", [(2731, 17, 3), (2048, 49, 4), (2731, 97, 3), (2731, 145, 3)])
def test_block_widths(isolir, shape):
    """8192 solves are the most that blocks of 32 columns take; 8193 fill 64-column
    blocks but for one column in the last. A term's solves have the bits of its
    one-term call (32 columns, against the oracle above) and the solar ones are
    compared with the oracle as well. (Not the infra-red ones: the oracle's spread
    is the largest of three random runs, which so many thin layers exceed now and
    then.)"""
    P, L, G = shape
    tsc = synth.make_two_stream_case(P, L, isolir, seed=70 + L + isolir, n_term=G, omc_range=(-3.0, 0.0))
    gpu = R.two_stream_case(tsc, "fp64")
    for g in range(G):
        term = synth.two_stream_term(tsc, g)
        one = R.two_stream_case(dict(term, **{k: term[k][None] for k in ("tau", "omega", "asymmetry")}), "fp64")
        for k in ("flux_up", "flux_down") + (("flux_direct",) if isolir == 1 else ()):
            assert np.array_equal(gpu[k][g], one[k][0]), (k, g)
    if isolir == 1:
        _check(gpu, _oracle_terms(tsc), None, "fp64 %s" % (shape,))


def test_more_solves_than_one_launch_holds():
    """2^28 + 2^14 solves take three launches; every term has the same inputs,
    so all have the bits of a one-term call."""
    import torch
    P, G = 1 << 14, (1 << 14) + 1
    tsc = synth.make_two_stream_case(P, 2, 2, seed=79, n_term=1, omc_range=(-3.0, 0.0))
    dev = {k: torch.as_tensor(v).cuda() if isinstance(v, np.ndarray) else v for k, v in tsc.items()}
    torch.cuda.synchronize()   # the library has a stream of its own
    one = R.two_stream_case(dev, "fp64")
    many = dict(dev, n_term=G, **{k: dev[k].reshape(1, 2, P).repeat(G, 1, 1) for k in ("tau", "omega", "asymmetry")})
    out = {k: torch.full((G, 3, P), float("nan"), dtype=torch.float64, device="cuda") for k in ("flux_up", "flux_down")}
    out["flux_direct"] = None
    torch.cuda.synchronize()
    R.two_stream_case(many, "fp64", out=out)
    for k in ("flux_up", "flux_down"):
        assert bool((out[k] == one[k].reshape(1, 3, P)).all()), k
