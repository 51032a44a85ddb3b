"""The candidate walk of the cell-list and naive kernels (a group of lanes per
particle, or one lane from 49152 particles on; touching candidates queued in
LDS) where it can go wrong: fewer particles than lanes, a last wavefront that
is nearly empty, several particles per lane group, grids with fewer than three cells per axis, stencils of more
columns than lanes, and packings so dense that the queue is flushed more than
once per particle.  Forces, torques and a few steps equal the oracle bit for
bit; energies are float64 sums (relative 1e-12)."""

from __future__ import annotations

import numpy as np
import pytest

import jaxdem_amd as jd
from jaxdem_amd.utils.contacts import compute_contact_stress_tensor
from oracle import jdem_oracle as O
from tests import oracle_bridge as B
from tests.test_gpu_parity import assert_bitwise, packed

pytestmark = pytest.mark.gpu

# collider, dim, domain, N, volume fraction, cell edge / largest diameter
CASES = [
    ("naive", 3, "reflect", 1, 0.5, None),
    ("naive", 2, "periodic", 63, 0.6, None),
    ("naive", 3, "periodic", 65, 40.0, None),  # every pair touches: the queue of 128 fills
    ("naive", 3, "reflect", 1025, 0.5, None),
    ("CellList", 3, "periodic", 2, 0.1, 1.0),
    ("CellList", 3, "periodic", 40, 0.6, 1.0),  # one or two cells per axis
    ("CellList", 2, "reflect", 127, 12.0, 1.0),
    ("CellList", 3, "periodic", 401, 8.0, 1.0),  # about a hundred contacts per sphere
    ("CellList", 3, "reflect", 1500, 0.5, 0.5),  # 25 columns of 5 cells
    ("CellList", 2, "periodic", 1500, 0.7, 0.34),  # 7 columns of 7 cells
    ("CellList", 2, "reflect", 30011, 0.7, 1.0),
    ("CellList", 2, "periodic", 66001, 0.7, 1.0),  # one lane per disk
    ("CellList", 2, "reflect", 49153, 6.0, 1.0),  # one lane per disk, its queue of 12 flushed early
    ("CellList", 3, "periodic", 49153, 0.4, 1.0),
]


@pytest.mark.parametrize("collider,dim,domain,N,phi,edge", CASES)
def test_forces_steps_and_energy(device, collider, dim, domain, N, phi, edge):
    print(f"[walk] {collider} dim={dim} {domain} N={N} phi={phi} edge={edge}", flush=True)
    st, box = packed(N, dim, seed=N + dim, domain=domain, phi=phi)
    mats = [jd.Material.create("elasticfrict", density=1.0, young=1e3, poisson=0.3, mu=0.4, e=0.7, mu_r=0.05)]
    ckw = dict(state=st, cell_size=float(edge) * 2.0 * float(st.rad.max())) if collider == "CellList" else {}
    sy = jd.System.create(st.shape, dt=1e-4, domain_type=domain, domain_kw=dict(box_size=box, anchor=np.zeros(dim)),
                          collider_type=collider, collider_kw=ckw, force_model_type="cundallstrack",
                          mat_table=jd.MaterialTable.from_materials(mats))
    P = B.params_of(st, sy)
    st2, _ = sy.collider.compute_force(st, sy)
    ost = B.state_of(st)
    O.compute_force(ost, P)
    assert_bitwise("force", st2.force.cpu().numpy(), ost.force)
    assert_bitwise("torque", st2.torque.cpu().numpy(), ost.torque)
    e, want = sy.potential_energy(st), O.potential_energy(B.state_of(st), P)
    assert abs(e - want) <= 1e-12 * abs(want)
    if collider == "naive":
        cand = O.naive_candidates(N)
    else:
        cand, _ = O.cell_candidates(B.state_of(st).pos, P.domain, P.cell_size, P.search_range)
    vir = O.pair_virial(B.state_of(st), P, cand) / float(np.prod(box.astype(np.float64)))
    got = compute_contact_stress_tensor(st, sy)[2]
    assert np.abs(got - vir).max() <= 1e-12 * np.abs(vir).max()
    n = 2 if N > 10000 else 4
    st3, _ = jd.System.step(st, sy, n=n)
    ost = O.step(B.state_of(st), P, n)
    assert_bitwise("pos", st3.pos_c.cpu().numpy(), ost.pos)
    assert_bitwise("vel", st3.vel.cpu().numpy(), ost.vel)
    assert_bitwise("ang_vel", st3.ang_vel.cpu().numpy(), ost.ang_vel)
