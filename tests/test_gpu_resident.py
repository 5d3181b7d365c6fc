"""Small :dipole replicas stepped inside one launch per call, against the
launch per stage on the same layout: sizes around one workgroup and around
the largest exchange, ragged parts, axes shorter than a bond, many
sublattices, and every kind of bond and onsite term.

Both run the same per-site arithmetic.  Seven Langevin or midpoint steps (or
eight, with the same bound, of the largest replicas) round about 7 x 20 times; with the spread of one rounding over the steps
(at most tenfold) that is 7 x 20 x 10 x 2^-53 = 1.6e-13 in FP64 and 8e-5 in
FP32, relative to |S|.
"""
import numpy as np
import pytest

import sunnyhip as sh

from helpers import announce, rel_err

pytestmark = pytest.mark.gpu

TOL = {64: 1.6e-13, 32: 8e-5}


def general_model(dims, precision):
    """Anisotropic exchange, biquadratic bonds, a field, Stevens terms to order 6."""
    s = sh.System(sh.cubic_crystal(1.0), [(0, sh.Moment(s=3, g=2))], "dipole", dims=dims, seed=5, precision=precision)
    J = np.array([[1.0, 0.2, -0.1], [0.1, 0.8, 0.05], [0.0, -0.2, 1.1]])
    sh.set_exchange_(s, J, sh.Bond(0, 0, (1, 0, 0)))
    sh.set_exchange_(s, 0.5, sh.Bond(0, 0, (0, 1, 0)), biquad=0.03,
                     propagate=[sh.Bond(0, 0, (0, 1, 0)), sh.Bond(0, 0, (0, 0, 1))])
    sh.set_onsite_coupling_(s, lambda S: 0.02 * S[2] @ S[2] @ S[2] @ S[2] +
                            0.001 * S[0] @ S[0] @ S[0] @ S[0] @ S[0] @ S[0], 0)
    sh.set_field_(s, [0.3, -0.1, 0.2])
    sh.randomize_spins_(s)
    return s


def inhomogeneous(dims, precision):
    """One sublattice per site (a vacancy among them): parts of a single cell."""
    s = sh.to_inhomogeneous(sh.workloads.cubic_model(dims=dims, seed=6, precision=precision))
    sh.set_vacancy_at_(s, (1, 0, 1, 0))
    return s


def build(kind, dims, precision):
    if kind == "cubic":
        return sh.workloads.cubic_model(dims=dims, seed=4, precision=precision)
    if kind == "pyrochlore":
        return sh.workloads.pyrochlore_model(dims=dims, seed=4, precision=precision)
    return {"general": general_model, "inhomogeneous": inhomogeneous}[kind](dims, precision)


@pytest.mark.parametrize("kind,dims,precision,layout", [
    ("cubic", (1, 1, 1), 64, 1),       # one site, bonded to itself
    ("cubic", (8, 8, 8), 64, 1),       # 512 sites: the largest single workgroup
    ("cubic", (27, 19, 1), 64, 1),     # 513 sites: the smallest that is cut
    ("cubic", (2, 1, 300), 64, 1),     # axes shorter than the parts
    ("cubic", (19, 17, 13), 32, 1),    # ragged parts
    ("cubic", (20, 20, 20), 64, 1),    # 125 parts
    ("cubic", (16, 16, 32), 32, 1),
    ("cubic", (28, 32, 32), 64, 1),    # 28672 sites: the most
    ("cubic", (27, 29, 31), 32, 0),    # tiled layout
    ("pyrochlore", (12, 11, 12), 32, 0),
    ("pyrochlore", (2, 3, 5), 64, 1),  # one workgroup, sixteen sublattices
    ("pyrochlore", (5, 3, 4), 64, 1),  # four cells a part
    ("pyrochlore", (8, 8, 8), 32, 1),
    ("general", (5, 6, 7), 64, 1),
    ("general", (11, 9, 8), 64, 1),
    ("general", (11, 9, 8), 32, 1),
    ("inhomogeneous", (9, 9, 9), 64, 1),
])
def test_resident_steps_match_launches(kind, dims, precision, layout, monkeypatch):
    announce(f"resident vs launched {kind} {dims} fp{precision} layout {layout}")

    def handle(on):
        monkeypatch.setenv("SNH_PERSIST", on)
        monkeypatch.setenv("SNH_COOP", on)
        s = build(kind, dims, precision)
        s.layout = layout
        h = s._device()
        assert h.query("layout") == layout
        assert h.query("persistent") + h.query("cooperative") == int(on)
        return s

    def resident(calls):
        h = a._device()
        assert h.query("resident_calls") == calls and h.query("persistent") + h.query("cooperative") == 1
        assert b._device().query("resident_calls") == 0

    a, b = handle("1"), handle("0")
    kap = float(np.max(a.kappas))
    lang = sh.Langevin(0.02 / kap, damping=0.1, kT=0.4)
    n = 7 if a.nsites < 20000 else 8  # from which the largest replicas step resident
    sh.step_(a, lang, nsteps=n)
    sh.step_(b, lang, nsteps=n)
    assert np.all(np.isfinite(b.dipoles_flat()))
    assert rel_err(a.dipoles_flat(), b.dipoles_flat(), scale=kap) <= TOL[precision]
    # the noise goes on where the call before ended
    sh.step_(a, lang, nsteps=n)
    sh.step_(b, lang, nsteps=n)
    assert rel_err(a.dipoles_flat(), b.dipoles_flat(), scale=kap) <= 2 * TOL[precision]
    resident(2)
    b.set_state_flat(dip=a.dipoles_flat())
    mid = sh.ImplicitMidpoint(0.01 / kap, damping=0.05, tol=1e-12 if precision == 64 else 1e-5)
    ia, ib = sh.step_(a, mid, nsteps=7), sh.step_(b, mid, nsteps=7)
    assert abs(int(ia[0]) - int(ib[0])) <= 1
    assert rel_err(a.dipoles_flat(), b.dipoles_flat(), scale=kap) <= TOL[precision] + mid.tol
    resident(3)


@pytest.mark.parametrize("kind,dims,precision,layout,least", [
    ("cubic", (27, 19, 1), 64, 1, 5),       # the smallest that is cut
    ("cubic", (16, 16, 32), 32, 1, 6),
    ("cubic", (27, 29, 31), 32, 0, 3),      # tiled layout
    ("cubic", (28, 32, 32), 64, 1, 8),      # 28672 sites: the most
    ("pyrochlore", (4, 3, 5), 64, 1, 5),
    ("pyrochlore", (12, 12, 12), 64, 1, 22),  # 18 bonds a site: a resident step gains little
    ("pyrochlore", (12, 11, 12), 32, 0, 3),
    ("general", (11, 9, 8), 64, 1, 5),
    ("general", (11, 9, 8), 32, 1, 5),
    ("inhomogeneous", (9, 9, 9), 32, 1, 5),
])
def test_langevin_calls_may_be_split_anywhere(kind, dims, precision, layout, least, monkeypatch):
    """Calls of few steps are launched, longer ones resident, and all calls
    launched while kernels are timed: the states are the same bit for bit
    however a run is cut into calls."""
    announce(f"split calls {kind} {dims} fp{precision} layout {layout}")
    monkeypatch.setenv("SNH_COOP", "1")

    def run(calls, timed=False, kT=0.4):
        s = build(kind, dims, precision)
        s.layout = layout
        h = s._device()
        assert h.query("layout") == layout
        kap = float(np.max(s.kappas))
        h.call("snh_enable_timing", int(timed))
        for n in calls:
            before = h.query("resident_calls")
            sh.step_(s, sh.Langevin(0.02 / kap, damping=0.1, kT=kT), nsteps=n)
            assert h.query("resident_calls") - before == int(n >= least and not timed)
        S = s.dipoles_flat()
        assert h.query("cooperative") == 1
        return S

    n = 2 * least + 3
    whole = run([n])
    assert np.all(np.isfinite(whole))
    np.testing.assert_array_equal(run([1, least, 1, least - 1, 2]), whole)
    np.testing.assert_array_equal(run([least - 1, n + 1 - least]), whole)
    np.testing.assert_array_equal(run([n], timed=True), whole)
    np.testing.assert_array_equal(run([n], kT=0.0), run([1] * n, kT=0.0))  # and without noise


@pytest.mark.parametrize("dims", [(6, 7, 9), (9, 10, 7)])  # one part; several
def test_calls_longer_than_a_launch(dims, monkeypatch):
    """4096 steps are one launch, the rest of the call the next: the noise and
    the exchanged words go on across them."""
    announce(f"9000 steps in a call {dims}")
    monkeypatch.setenv("SNH_PERSIST", "1")
    monkeypatch.setenv("SNH_COOP", "1")
    lang = sh.Langevin(0.05, damping=0.1, kT=0.4)
    out = []
    for calls in ([9000], [4096, 4096, 808], [5000, 4000]):
        s = build("cubic", dims, 64)
        s.layout = 1
        for n in calls:
            sh.step_(s, lang, nsteps=n)
        out.append(s.dipoles_flat())
        assert s._device().query("resident_calls") == len(calls)
        assert s._device().query("persistent") + s._device().query("cooperative") == 1
    np.testing.assert_array_equal(out[1], out[0])
    np.testing.assert_array_equal(out[2], out[0])
    monkeypatch.setenv("SNH_PERSIST", "0")
    monkeypatch.setenv("SNH_COOP", "0")
    s = build("cubic", dims, 64)
    s.layout = 1
    sh.step_(s, lang, nsteps=9000)
    np.testing.assert_array_equal(s.dipoles_flat(), out[0])


def test_handles_of_several_threads():
    """Four replicas of 432 parts each, more than the device holds side by
    side, step on four threads: every launch finds its parts resident, and the
    states are those of one thread."""
    import threading

    announce("resident handles on four threads")
    lang, mid = sh.Langevin(0.02, damping=0.1, kT=0.3), sh.ImplicitMidpoint(0.02)

    def models():
        out = [sh.workloads.pyrochlore_model(L=12, seed=40 + r, precision=64) for r in range(4)]
        for s in out:
            assert s._device().query("cooperative") == 1
        return out

    def work(s):
        for _ in range(3):
            sh.step_(s, lang, nsteps=40)
            sh.step_(s, mid, nsteps=2)

    one = models()
    for s in one:
        work(s)
    many = models()
    threads = [threading.Thread(target=work, args=(s,)) for s in many]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(one, many):
        assert b._device().query("resident_calls") == 6 and b._device().query("cooperative") == 1
        np.testing.assert_array_equal(b.dipoles_flat(), a.dipoles_flat())


def next_calls():
    """What a program may do after a Langevin call: reads of the state, and
    everything that changes it."""
    lang, mid = sh.Langevin(0.03, damping=0.2, kT=0.7), sh.ImplicitMidpoint(0.02, damping=0.1)
    sampler = sh.LocalSampler(kT=0.4, nsweeps=1.5)
    return {
        "spins": lambda s: None,
        "energy": sh.energy,
        "gradient": sh.energy_grad_dipoles,
        "synchronize": lambda s: s._device().call("snh_synchronize"),
        "steps": lambda s: sh.step_(s, lang, nsteps=3),
        "midpoint": lambda s: sh.step_(s, mid, nsteps=2),
        "sampler": lambda s: sh.step_(s, sampler),
    }


@pytest.mark.parametrize("after", list(next_calls()))
def test_lost_parts_leave_the_launched_result(after, monkeypatch):
    """Parts that give up waiting (here at the first word that is not there
    yet) must not cost the state: the call is made again by launches, whatever
    comes next, and the handle keeps to them."""
    announce(f"lost Langevin parts, then {after}")

    def run(coop, spin):
        monkeypatch.setenv("SNH_COOP", coop)
        monkeypatch.setenv("SNH_RES_SPIN", spin)
        s = sh.workloads.cubic_model(L=16, seed=7, precision=64)
        s.layout = 1
        assert s._device().query("cooperative") == int(coop)
        sh.step_(s, sh.Langevin(0.05, damping=0.1, kT=0.5), nsteps=40)
        out = next_calls()[after](s)
        first = s.dipoles_flat()
        s._dev_dirty = True
        np.testing.assert_array_equal(s.dipoles_flat(), first)  # a second read
        return s, out, first

    a, oa, Sa = run("1", "0")
    b, ob, Sb = run("0", "0")
    assert a._device().query("cooperative") == 0
    np.testing.assert_array_equal(Sa, Sb)
    if ob is not None:
        np.testing.assert_array_equal(oa, ob)
    a.set_state_flat(dip=Sa[::-1].copy())  # and a new state is taken as ever
    sh.energy(a)
    a._dev_dirty = True
    np.testing.assert_array_equal(a.dipoles_flat(), Sa[::-1])


def test_lost_midpoint_parts_leave_the_launched_result(monkeypatch):
    announce("lost midpoint parts")

    def make(coop):
        monkeypatch.setenv("SNH_COOP", coop)
        monkeypatch.setenv("SNH_RES_SPIN", "0")
        s = sh.workloads.cubic_model(L=16, seed=7, precision=64)
        s.layout = 1
        s._device()
        return s

    a, b = make("1"), make("0")
    mid = sh.ImplicitMidpoint(0.02, damping=0.1)
    np.testing.assert_array_equal(sh.step_(a, mid, nsteps=5), sh.step_(b, mid, nsteps=5))
    assert a._device().query("cooperative") == 0
    np.testing.assert_array_equal(a.dipoles_flat(), b.dipoles_flat())
    # a trajectory's recording loses its first step and goes on by launches
    w = np.arange(3.0 * a.nsites).reshape(-1, 3)
    grads = [sh.midpoint_gradient(s, sh.ImplicitMidpoint(0.02), 4, [], lambda S: (float((w * S).sum()), w))
             for s in (make("1"), make("0"))]
    for x, y in zip(*grads):
        np.testing.assert_array_equal(x, y)


def test_energy_read_from_lost_parts_is_reported(monkeypatch):
    """An energy queued without waiting reads a lost call's spins before the
    call is made again: the next waiting call says so, once, and the state is
    the launched one."""
    announce("lost parts, energy without waiting")
    from test_zz_no_alloc import noalloc_energy

    def make(coop):
        monkeypatch.setenv("SNH_COOP", coop)
        monkeypatch.setenv("SNH_RES_SPIN", "0")
        s = sh.workloads.cubic_model(L=16, seed=7, precision=64)
        s.layout = 1
        sh.step_(s, sh.Langevin(0.05, damping=0.1, kT=0.5), nsteps=40)
        return s

    a, b = make("1"), make("0")
    with pytest.raises(RuntimeError, match="made again"):
        noalloc_energy(a)
    np.testing.assert_array_equal(noalloc_energy(a), noalloc_energy(b))
    np.testing.assert_array_equal(a.dipoles_flat(), b.dipoles_flat())
