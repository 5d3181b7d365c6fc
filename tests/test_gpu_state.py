"""Setting and reading back states: the device's copy of a state is the host's,
rounded to the device's precision and no further, for transfers of one chunk
and of several, both layouts, uneven batches, axes shorter than the longest
bond (ghost images that wrap more than once) and kets of every N; a ket's
dipole is its expected spin in FP64 (a few hundred roundings: 1e-13); and
the energy of an uploaded state, which reads the ghost images, is the
oracle's."""
import numpy as np
import pytest

import sunnyhip as sh
from oracle import oracle as O

from helpers import announce, energy_scale

pytestmark = pytest.mark.gpu


def fresh(s):
    """Reads the state back from the device (the host's copy is overwritten)."""
    sh.energy(s)
    (s._coh if s.N else s._dip)[:] = np.nan
    s._dev_dirty = True
    return s.coherents_flat() if s.N else s.dipoles_flat()


def rounded(x, precision):
    return x if precision == 64 else x.astype(np.complex64 if np.iscomplexobj(x) else np.float32).astype(x.dtype)


@pytest.mark.parametrize("model,dims,precision,layout", [
    ("cubic", (1, 1, 1), 64, 1),
    ("cubic", (5, 1, 2), 32, 1),
    ("cubic", (64, 64, 64), 64, 1),   # two chunks
    ("cubic", (97, 61, 59), 32, 0),   # one chunk and a ragged rest
    ("pyrochlore", (1, 2, 1), 64, 1),
    ("pyrochlore", (13, 11, 9), 32, 0),
    ("pyrochlore", (13, 11, 9), 32, 1),
])
def test_dipole_state_round_trip(model, dims, precision, layout):
    announce(f"state {model} {dims} fp{precision} layout {layout}")
    make = sh.workloads.cubic_model if model == "cubic" else sh.workloads.pyrochlore_model
    s = make(dims=dims, seed=8, precision=precision)
    s.layout = layout
    S = s.dipoles_flat()
    E = sh.energy(s)
    np.testing.assert_array_equal(fresh(s), rounded(S, precision))
    if s.nsites < 30000:
        assert abs(E - O.Oracle(s.spec()).energy(S)) <= (1e-11 if precision == 64 else 1e-5) * energy_scale(s)


@pytest.mark.parametrize("N", [2, 3, 5, 7])
@pytest.mark.parametrize("precision", [64, 32])
def test_ket_state_round_trip(N, precision):
    announce(f"state SU({N}) fp{precision}")
    s = sh.workloads.triangular_sun_model(L1=7, L2=2, s=(N - 1) / 2, D=0.0 if N == 2 else 0.4, seed=9,
                                          precision=precision)
    Z = rounded(s.coherents_flat(), precision)
    np.testing.assert_array_equal(fresh(s), Z)
    np.testing.assert_allclose(s.dipoles_flat(), sh.expected_spin_host(Z, N), rtol=0, atol=1e-13)


def test_uneven_batches_round_trip():
    announce("state of uneven batches")
    systems = [sh.workloads.triangular_sun_model(L1=L, seed=20 + L, precision=32) for L in (5, 300, 64, 1)]
    kets = [rounded(s.coherents_flat(), 32) for s in systems]
    b = sh.ReplicaBatch(systems, precision=32)
    sh.energy(b)
    b._dev_dirty = True
    b.sync_to_systems()
    for s, Z in zip(systems, kets):
        np.testing.assert_array_equal(s.coherents_flat(), Z)
        np.testing.assert_allclose(s.dipoles_flat(), sh.expected_spin_host(Z, 3), rtol=0, atol=1e-13)
    systems = [sh.workloads.cubic_model(dims=d, seed=30 + d[0], precision=32) for d in ((80, 70, 60), (3, 1, 2), (9, 8, 7))]
    dips = [rounded(s.dipoles_flat(), 32) for s in systems]
    b = sh.ReplicaBatch(systems, precision=32)
    sh.energy(b)
    b._dev_dirty = True
    b.sync_to_systems()
    for s, S in zip(systems, dips):
        np.testing.assert_array_equal(s.dipoles_flat(), S)
        s.set_state_flat(dip=S)  # the systems' own copies are independent of the batch
    b._dev_dirty = True
    b.sync_to_systems()
    np.testing.assert_array_equal(systems[2].dipoles_flat(), dips[2])
