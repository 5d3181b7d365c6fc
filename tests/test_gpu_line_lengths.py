"""Every length of the transforms' lines, along every axis, against the
oracle's Ewald energy and gradient: lengths transformed in registers (factors
2, 3, 4, 5, 7, 11, 13 and their products), the primes beyond, and the widths
of a line's half spectrum, even and odd.  FP64 agrees to rounding (the same
1e-11 as the other Ewald parity tests), FP32 to 2e-5.  A batch large enough
for three fields a workgroup takes every replica through that form."""
import numpy as np
import pytest

import sunnyhip as sh
from oracle import oracle as O

from helpers import announce, rel_err

pytestmark = pytest.mark.gpu


def dipolar(dims, precision, seed):
    s = sh.workloads.cubic_model(dims=dims, J=0.3, D=0.0, seed=seed, precision=precision)
    sh.enable_dipole_dipole_(s, 0.7)
    return s


@pytest.mark.parametrize("precision,tol", [(64, 1e-11), (32, 2e-5)])
@pytest.mark.parametrize("L", range(1, 33))
def test_line_lengths(L, precision, tol, monkeypatch):
    for axis in range(3):
        dims = [2, 3, 2]
        dims[axis] = L
        for slab in ("0", "1"):  # one workgroup per field; axes split
            announce(f"lines of {L} along axis {axis} fp{precision} slab {slab}")
            monkeypatch.setenv("SNH_EWALD_SLAB", slab)
            s = dipolar(tuple(dims), precision, seed=L)
            o = O.Oracle(s.spec())
            S = s.dipoles_flat()
            g = o.grad(S)
            assert rel_err(sh.energy_grad_dipoles(s), g) <= tol
            assert abs(sh.energy(s) - o.energy(S)) <= tol * np.abs(g * S).sum()


@pytest.mark.parametrize("dims", [(5, 3, 4), (8, 7, 2), (16, 3, 2), (3, 2, 16)])
def test_three_fields_a_workgroup(dims):
    announce(f"three fields {dims}")
    one = sh.workloads.pyrochlore_model(dims=dims, J1=0.05, J2=0.0, A=0.0, s=3.5, seed=3, precision=32, dipolar=True)
    systems = [sh.clone_system(one, seed=r) for r in range(16)]
    for s in systems:
        sh.randomize_spins_(s)
    b = sh.ReplicaBatch(systems, precision=32)
    h = b._device()
    g = np.empty((h.total, 3))
    h.call("snh_energy_grad", sh._lib.dptr(g))
    n = one.nsites
    for r in (0, 7, 15):
        assert rel_err(g[r * n:(r + 1) * n], O.Oracle(one.spec()).grad(systems[r].dipoles_flat())) <= 2e-5


@pytest.mark.parametrize("dims", [(5, 3, 4), (2, 16, 2)])
def test_three_fields_with_the_potential_in_fp64(dims):
    """The batch's Metropolis trials refresh their FP64 potential by the same
    transforms after every 512 trials: the energy changes they add up are the
    oracle's energy differences, to 2e-5 of a full turn in the largest local
    field for each trial."""
    announce(f"three fields, FP64 potential {dims}")
    one = sh.workloads.pyrochlore_model(dims=dims, J1=0.05, J2=0.0, A=0.0, s=3.5, seed=5, precision=32, dipolar=True)
    systems = [sh.clone_system(one, seed=r) for r in range(16)]
    for s in systems:
        sh.randomize_spins_(s)
    o = O.Oracle(one.spec())
    before = [s.dipoles_flat() for s in systems]
    b = sh.ReplicaBatch(systems, precision=32)
    sampler = sh.LocalSampler(kT=2.0, nsweeps=1.0)
    sh.step_(b, sampler)
    b.sync_to_systems()
    assert one.nsites > 512
    for r in (0, 7, 15):
        after = systems[r].dipoles_flat()
        turn = 2 * 3.5 * np.max(np.linalg.norm(o.grad(before[r]), axis=1))
        assert abs(sampler.dE[r] - (o.energy(after) - o.energy(before[r]))) <= 2e-5 * one.nsites * turn
        assert np.count_nonzero(np.any(after != before[r], axis=1)) > one.nsites // 10
