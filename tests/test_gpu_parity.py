"""Parity of the HIP hydro step with the FP64 oracle, through the C ABI.

Both sides start from the same host initial state (InitGasDensity with the
drand48 noise stream, InitEuler), take AlgoGas calls of the same DT and are
compared field by field.  Bars:
  * integer work is bit-exact: FARGO shifts Nshift[i], the number of CFL
    sub-steps per call;
  * FP64 fields: relative L-infinity error (max |gpu - oracle| / max |oracle|)
    <= 1e-12 after a few calls and <= 1e-11 after 10 orbits, for Sigma,
    v_theta and energy; the radial velocity is measured on the velocity
    scale max |v_theta| with the same bars;
  * FP32 storage: <= 2e-5 (Sigma), 2e-6 (velocities) after a few calls.
Differences come only from reduction order (ring means, force sums, FFT), as
pointwise arithmetic is the reference's, built without contraction.
"""
import math

import numpy as np
import pytest

from dustyfargoadsg_amd import _capi
from dustyfargoadsg_amd.disc import Disc, DfargoError
from dustyfargoadsg_amd.workloads import gas_planet, energy_sg
from tests.oracle_lib import Oracle

pytestmark = pytest.mark.gpu

DT = 2 * math.pi / 20  # one .par DT: twenty per orbit at r = 1


def rel(a, b, nr, ns):
    a, b = a[: nr * ns], b[: nr * ns]
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def pair(params, planets, precision=_capi.FP64):
    print(f"case {params.nrad}x{params.nsec} prec={precision}", flush=True)
    o = Oracle(params)
    so = o.initial_state(planets)
    d = Disc(params, precision)
    sg = d.initial_state(planets)
    return o, so, d, sg


def compare(o, d, p, tol_rho, tol_vr, tol_vt, tol_e=None):
    """vr is compared on the velocity scale max|v_theta|: its own maximum is
    ~1e-3 of that, so a max|vr|-relative figure would mostly measure how
    small vr is."""
    go, oo = d.state(), o.state()
    errs = {k: rel(go[k], oo[k], p.nrad, p.nsec) for k in ("rho", "vt", "energy")}
    n = p.nrad * p.nsec
    errs["vr"] = np.abs(go["vr"][:n] - oo["vr"][:n]).max() / np.abs(oo["vt"][:n]).max()
    errs["vr_own_scale"] = rel(go["vr"], oo["vr"], p.nrad, p.nsec)
    assert errs["rho"] <= tol_rho, errs
    assert errs["vr"] <= tol_vr, errs
    assert errs["vt"] <= tol_vt, errs
    if p.energy_equation:
        assert errs["energy"] <= (tol_e or tol_rho), errs
    return errs, go, oo


# the 1536- and 3072-cell rings take the six-cells-per-thread launches of the
# ring kernels (K = 6) that the full-size discs use
@pytest.mark.parametrize("nr,ns,calls", [(32, 96, 3), (128, 384, 2), (16, 1536, 1), (16, 3072, 1)])
def test_gas_planet_fp64(nr, ns, calls):
    p, pl = gas_planet(nrad=nr, nsec=ns)
    o, so, d, sg = pair(p, pl)
    for k in ("rho", "vr", "vt"):
        assert np.array_equal(sg[k], so[k]), k
    for c in range(calls):
        n_o = o.algogas(DT)
        d.algogas(DT)
        st, sto = d.status(), o.status()
        assert st.last_call_substeps == n_o
        nsh_g, vm_g = d.fargo_shift()
        nsh_o, vm_o = o.fargo_shift()
        assert np.array_equal(nsh_g, nsh_o)
        assert np.abs(vm_g - vm_o).max() <= 1e-13 * np.abs(vm_o).max()
        assert abs(st.physical_time - sto.physical_time) <= 1e-15
        assert abs(st.lost_mass - sto.lost_mass) <= 1e-10 * abs(sto.lost_mass)
    errs, go, oo = compare(o, d, p, 1e-12, 1e-12, 1e-12)
    assert abs(go["planets"].x[0] - oo["planets"].x[0]) <= 1e-14
    assert abs(go["planets"].y[0] - oo["planets"].y[0]) <= 1e-14


# rings whose threads (one to four cells each) are no whole number of
# wavefronts, with a planet that feels the disc: the ring reductions at their
# remainders, the n-body step with a free planet.  The file's FP64 bars.
@pytest.mark.parametrize("ns", [8, 63, 97, 400, 1030, 1530, 1533, 2044])
@pytest.mark.parametrize("energy", [0, 1])
def test_ragged_rings_fp64(ns, energy):
    p, pl = gas_planet(nrad=12, nsec=ns, forced_circular=0, energy_equation=energy, beta_cooling=energy)
    pl = dict(pl, feel_disk=[1])
    o, so, d, sg = pair(p, pl)
    n_o = o.algogas(DT)
    d.algogas(DT)
    assert d.status().last_call_substeps == n_o
    errs, go, oo = compare(o, d, p, 1e-12, 1e-12, 1e-12)
    for k in ("x", "y", "vx", "vy"):
        assert abs(getattr(go["planets"], k)[0] - getattr(oo["planets"], k)[0]) <= 1e-13, k


# Rings of 8, 12 and 16 cells a thread whose threads are no whole number of
# wavefronts, with the energy equation: there the CFL kernel reads the previous
# sound speed after its reduction and replaces it, each thread in its own cells
# alone.  Hot columns pass through column 0, the cell of which a thread past the
# ring would take the sound speed from either side of the replacement.  Twice,
# bit for bit, and the time steps, their number and the fields against the
# oracle with the file's bars.
@pytest.mark.parametrize("ns", [2056, 2080, 3200, 4104, 6176])
def test_ragged_wide_rings_fp64(ns):
    p, pl = gas_planet(nrad=8, nsec=ns, rmin=0.9, rmax=1.1, energy_equation=1, beta_cooling=1)
    o, so, d, sg = pair(p, pl)
    for st in (so, sg):
        e, vt = st["energy"].reshape(-1, ns), st["vt"].reshape(-1, ns)
        e[:, -8:] *= np.linspace(1.5, 4.0, 8)
        vt[:, -4:] += 0.01
    o.set_state(so)
    got = []
    for _ in range(2):
        d.set_state(sg)
        d.algogas(DT / 10)
        st = d.state()
        got.append((d.status().last_call_substeps, d.status().mindt, st["rho"], st["vr"], st["vt"], st["energy"]))
    n_o = o.algogas(DT / 10)
    assert got[0][0] == got[1][0] == n_o and n_o >= 3
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(a, b)
    assert abs(got[0][1] - o.status().mindt) <= 1e-12 * o.status().mindt
    compare(o, d, p, 1e-12, 1e-12, 1e-12)


# strips of more than one ring, the last of them shorter, on either side of
# the size from which the wavefronts outnumber the SIMDs.  The file's bars.
@pytest.mark.parametrize("nr", [41, 100])
@pytest.mark.parametrize("energy", [0, 1])
def test_strips_of_rings_fp64(nr, energy):
    p, pl = gas_planet(nrad=nr, nsec=3072, energy_equation=energy, beta_cooling=energy)
    o, so, d, sg = pair(p, pl)
    n_o = o.algogas(DT / 20)
    d.algogas(DT / 20)
    assert d.status().last_call_substeps == n_o
    compare(o, d, p, 1e-12, 1e-12, 1e-12)


@pytest.mark.parametrize("nr,ns,calls", [(32, 96, 2), (64, 192, 1), (16, 1536, 1), (16, 3072, 1)])
def test_energy_sg_fp64(nr, ns, calls):
    p, pl = energy_sg(nrad=nr, nsec=ns)
    o, so, d, sg = pair(p, pl)
    assert rel(sg["vt"], so["vt"], nr, ns) <= 1e-14
    for c in range(calls):
        n_o = o.algogas(DT)
        d.algogas(DT)
        assert d.status().last_call_substeps == n_o
        assert np.array_equal(d.fargo_shift()[0], o.fargo_shift()[0])
    compare(o, d, p, 1e-12, 1e-12, 1e-12, 1e-12)
    for f in ("divv", "vischeat", "sg_accr", "sg_acct"):
        assert rel(d.field(f), o.field(f), nr, ns) <= 1e-10, f


def test_sg_acceleration_matches_oracle():
    p, pl = energy_sg(nrad=64, nsec=192)
    o, so, d, sg = pair(p, pl)
    ar, at = d.compute_selfgravity()
    ar_o, at_o = o.sg_accel(so["rho"])
    assert rel(ar, ar_o, 64, 192) <= 1e-13
    assert rel(at, at_o, 64, 192) <= 1e-11


@pytest.mark.parametrize("variant", ["open", "standard", "feel_disk", "taper", "no_indirect", "discard_gas_indirect",
                                     "alternative_gas_indirect"])
def test_parameter_variants_fp64(variant):
    """Boundary, transport and planet options against the oracle."""
    if variant == "feel_disk":
        p, pl = gas_planet(nrad=32, nsec=96, forced_circular=0)
        pl = dict(pl, feel_disk=[1], feel_others=[1])
    elif variant == "taper":
        p, pl = gas_planet(nrad=32, nsec=96, forced_circular=0, mass_taper=0.5)
        pl = dict(pl, feel_disk=[1], feel_others=[0])
    else:
        over = {"open": dict(boundary=_capi.BC_OPEN), "standard": dict(fast_transport=0),
                "no_indirect": dict(indirect_term=0), "discard_gas_indirect": dict(discard_gas_indirect_term=1),
                "alternative_gas_indirect": dict(alternative_gas_indirect_term=1)}[variant]
        p, pl = gas_planet(nrad=32, nsec=96, **over)
    o, so, d, sg = pair(p, pl)
    for _ in range(2):
        n_o = o.algogas(DT)
        d.algogas(DT)
        assert d.status().last_call_substeps == n_o
        assert np.array_equal(d.fargo_shift()[0], o.fargo_shift()[0])
    errs, go, oo = compare(o, d, p, 1e-12, 1e-12, 1e-12)
    for k in ("x", "y", "vx", "vy", "mass"):
        assert abs(getattr(go["planets"], k)[0] - getattr(oo["planets"], k)[0]) <= 1e-13, k


def test_fp32_storage_within_bound():
    p, pl = gas_planet(nrad=128, nsec=384)
    o, so, d, sg = pair(p, pl, _capi.FP32)
    for _ in range(2):
        n_o = o.algogas(DT)
        d.algogas(DT)
        assert d.status().last_call_substeps == n_o
    compare(o, d, p, 2e-5, 2e-6, 2e-6)


@pytest.mark.parametrize("nr,ns", [(32, 96), (64, 192)])
def test_energy_sg_fp32_storage(nr, ns):
    """The benchmark's FP32 half: adiabatic self-gravitating disc with FP32
    storage, whose self-gravity transforms compute in float, against the
    FP64 oracle after two calls.  Bars: 2e-5 of max Sigma and max e, 2e-6 of
    max v_theta for both velocities (the planet-disc FP32 bars); the SG
    accelerations in float within 1e-5 of max |g_r| (g_theta, which only the
    1e-3 density noise makes, ~1e-3 of g_r, is measured on the g_r scale as
    v_r is on the v_theta scale); the same sub-step counts.  The integer FARGO shifts must match wherever the oracle's
    argument lies further than 1e-4 from a rounding tie (the float state
    moves the ring means by ~1e-7)."""
    p, pl = energy_sg(nrad=nr, nsec=ns)
    o, so, d, sg = pair(p, pl, _capi.FP32)
    ar, at = d.compute_selfgravity()
    ar_o, at_o = o.sg_accel(so["rho"])
    n = nr * ns
    gscale = np.abs(ar_o[:n]).max()
    errs = (rel(ar, ar_o, nr, ns), np.abs(at[:n] - at_o[:n]).max() / gscale)
    print("start-up SG accel (g_r, g_theta on the g_r scale) rel err", errs, flush=True)
    assert errs[0] <= 1e-5 and errs[1] <= 1e-5
    for c in range(2):
        n_o = o.algogas(DT)
        d.algogas(DT)
        assert d.status().last_call_substeps == n_o
        if o.status().fargo_margin > 1e-4:
            assert np.array_equal(d.fargo_shift()[0], o.fargo_shift()[0])
    errs, _, _ = compare(o, d, p, 2e-5, 2e-6, 2e-6, 2e-5)
    print("fp32 energy+sg errors", errs, flush=True)
    gr_o = o.field("sg_accr")
    assert rel(d.field("sg_accr"), gr_o, nr, ns) <= 1e-5
    assert np.abs(d.field("sg_acct")[:n] - o.field("sg_acct")[:n]).max() <= 1e-5 * np.abs(gr_o[:n]).max()


def test_graph_replay_equals_eager():
    """The sub-step graph replayed and the same kernels launched eagerly
    (profiling mode) give bit-identical states."""
    p, pl = energy_sg(nrad=32, nsec=96)
    d1, d2 = Disc(p), Disc(p)
    d1.initial_state(pl)
    d2.initial_state(pl)
    d2.set_profiling(True)
    for _ in range(3):
        d1.algogas(DT)
        d2.algogas(DT)
    s1, s2 = d1.state(), d2.state()
    for k in ("rho", "vr", "vt", "energy"):
        assert np.array_equal(s1[k], s2[k]), k
    times = d2.kernel_times()
    assert "transport_azi" in times and times["transport_azi"][1] > 0


def test_host_arrays_round_trip():
    """AlgoGas with host arrays (upload, step, download) equals the
    device-resident call."""
    p, pl = gas_planet(nrad=32, nsec=96)
    d1, d2 = Disc(p), Disc(p)
    st = d1.initial_state(pl)
    d2.initial_state(pl)
    d1.algogas(DT, state=st)
    d2.algogas(DT)
    s2 = d2.state()
    for k in ("rho", "vr", "vt"):
        assert np.array_equal(st[k], s2[k]), k
    assert st["planets"].x[0] == s2["planets"].x[0]


def test_run_substeps_exact_count_and_errors():
    p, pl = gas_planet(nrad=32, nsec=96)
    d = Disc(p)
    with pytest.raises(DfargoError):
        d.algogas(DT)  # before InitEuler
    d.initial_state(pl)
    d.run_substeps(1e6, 5)
    assert d.status().last_call_substeps == 5
    with pytest.raises(DfargoError):
        d.algogas(-1.0)


def test_gas_planet_ten_orbits_fp64():
    """The 128x384 planet disc over 10 orbits (200 AlgoGas calls): every
    field within 1e-11 of the oracle and every FARGO shift identical."""
    p, pl = gas_planet()
    o, so, d, sg = pair(p, pl)
    for c in range(200):
        o.algogas(DT)
        d.algogas(DT)
        if c % 20 == 19:
            assert np.array_equal(d.fargo_shift()[0], o.fargo_shift()[0]), c
            print(f"call {c + 1}", flush=True)
        # the FARGO shift's argument (Ntilde ~ 1-10) stays far from a
        # rounding tie compared with the ~1e-15 the ring-mean summation
        # order moves it; the margin itself agrees with the oracle's
        mg, mo = d.status().fargo_margin, o.status().fargo_margin
        assert abs(mg - mo) <= 1e-12 and mg > 1e-10, (mg, mo)
    assert d.status().substeps_total == o.status().substeps_total
    errs, _, _ = compare(o, d, p, 1e-11, 1e-11, 1e-11)
    print("10-orbit errors", errs, flush=True)
