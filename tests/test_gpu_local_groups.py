"""The packing of a workgroup's tried sites: colour classes of one site, just
under, at and past one workgroup's 256 sites, passes that try few of them, a
bond as long as an axis (the farthest the cheap neighbour index reaches), and
anisotropic bonds, against the oracle's trials with the same draws, which
FP64 follows to 1e-12 as in the other Metropolis tests."""
import numpy as np
import pytest

import sunnyhip as sh
from oracle import oracle as O

from helpers import announce

pytestmark = pytest.mark.gpu


def model(kind, dims):
    s = sh.workloads.cubic_model(dims=dims, seed=5, precision=64)
    if kind == "long":
        sh.set_exchange_(s, 0.3, sh.Bond(0, 0, (dims[0], 1, 0)), propagate=[sh.Bond(0, 0, (dims[0], 1, 0))])
    if kind == "aniso":
        J = np.array([[1.0, 0.2, -0.1], [0.1, 0.8, 0.05], [0.0, -0.2, 1.1]])
        sh.set_exchange_(s, J, sh.Bond(0, 0, (0, 1, 1)))
    sh.randomize_spins_(s)
    return s


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("kind,dims,nsweeps", [
    ("iso", (2, 2, 2), 1.0),      # classes of one site
    ("iso", (6, 10, 34), 1.0),    # 255 sites
    ("iso", (8, 16, 16), 1.5),    # 256
    ("iso", (2, 2, 514), 0.26),   # 257; the last pass tries one site in fifty
    ("long", (4, 6, 8), 1.0),
    ("aniso", (6, 10, 34), 1.0),
])
def test_packed_trials_match_oracle(kind, dims, nsweeps, layout):
    announce(f"packed trials {kind} {dims} nsweeps {nsweeps} layout {layout}")
    s = model(kind, dims)
    s.layout = layout
    prop = sh.propose_delta(0.4)
    S0 = s.dipoles_flat()
    m, nc, col = sh.local_coloring(s)
    ref, acc = O.Oracle(s.spec()).local_sweeps(S0, m, col.reshape(-1), nc, [(k, w, p) for k, w, p in prop.terms], 0.7,
                                               O.replica_key(s.noise_seed, 0), s.step_counter, nsweeps)
    sampler = sh.LocalSampler(kT=0.7, nsweeps=nsweeps, propose=prop)
    sh.step_(s, sampler)
    S = s.dipoles_flat()
    assert np.any(S != S0)
    assert np.max(np.abs(S - ref)) <= 1e-12
    np.testing.assert_allclose([sampler.dE, *sampler.dS], acc, rtol=0, atol=1e-11 * s.nsites)
