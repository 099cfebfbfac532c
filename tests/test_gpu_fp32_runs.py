"""FP32 storage against recorded runs.

A stored FP32 value is the FP64 result of the reference's operations in their
order, rounded by its own draw; the same kernels in another form must give the
same values.  Nothing weaker will do for particles that take the nearest
cell's values: a cell that rounds the other way moves a grain across an edge,
where it reads another cell and drags on that one, and within some hundred
sub-steps the Stokes numbers of the two runs differ by 4e-4 (64 x 150 cells,
10^4 grains, three calls).

tests/data/fp32_runs.npz was recorded from the kernels with the two transport
directions and the source terms in passes of their own.  Bar: equal bits in
all but 1 % of the values.  An ulp of FP64 (another order of a ring's sum,
another libm) turns one stored value in 2^29, none of the 10^6 of these runs;
1 % is the cells around one such value after the remaining sub-steps.
"""
import math
import os

import numpy as np
import pytest

from dustyfargoadsg_amd import _capi
from dustyfargoadsg_amd.disc import Disc, init_dust_system
from dustyfargoadsg_amd.workloads import energy_sg, gas_dust, gas_dust_particles

pytestmark = pytest.mark.gpu

DT = 2 * math.pi / 20
RECORDED = os.path.join(os.path.dirname(__file__), "data", "fp32_runs.npz")


def run(name):
    """The fields (FP32) and particles (FP64) after 25 sub-steps."""
    grains = name == "nearest_cell"
    p, pl = gas_dust(nrad=24, nsec=70) if grains else energy_sg(nrad=24, nsec=70, self_gravity=0)
    d = Disc(p, _capi.FP32)
    d.initial_state(pl)
    if grains:
        dp = gas_dust_particles(p, 500, seed=5, interpolation=_capi.INTERP_NGP, sizeminpart=1e-3)
        d.attach_dust(dp, init_dust_system(p, dp), DT)
    d.run_substeps(10 * DT, 25)
    st = d.state()
    out = {k: st[k].astype(np.float32) for k in ("rho", "vr", "vt") + (() if grains else ("energy",))}
    if grains:
        q = d.dust_state()
        out.update(grain_r=q["r"], grain_vr=q["vr"], grain_stokes=q["stokesnb"])
    return out


@pytest.mark.parametrize("name", ["nearest_cell", "energy"])
def test_fp32_run_is_the_recorded_one(name):
    print(f"case {name} 24x70 FP32, 25 sub-steps", flush=True)
    got, want = run(name), np.load(RECORDED)
    for k, x in got.items():
        y = want[f"{name}.{k}"]
        assert x.shape == y.shape and x.dtype == y.dtype
        assert np.mean(x != y) <= 0.01, (k, np.mean(x != y), np.abs(x - y).max())
