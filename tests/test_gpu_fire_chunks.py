"""The FIRE loop decided on the device: step limits and stops that fall inside
and on the edges of its chunks of iterations, particles that end inside a
block, gravity, fixed spheres: steps, positions, orientations and forces equal
the float32 oracle's, where further iterations were launched past the stop."""

from __future__ import annotations

import numpy as np
import pytest

import jaxdem_amd as jd
from jaxdem_amd import _lib as L
from oracle import jdem_oracle as O
from tests import oracle_bridge as B
from tests.test_gpu_parity import assert_bitwise, packed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,N,collider,max_steps,pe_diff_tol", [
    (3, 1, "naive", 3, -1.0),
    (2, 256, "naive", 4, -1.0),
    (3, 257, "CellList", 0, -1.0),
    (3, 257, "CellList", 5, -1.0),
    (3, 700, "CellList", 500, 5e-3),  # stops by itself, inside a chunk
    (2, 513, "NeighborList", 21, -1.0),
    (2, 900, "NeighborList", 500, 5e-4),
])
def test_chunks_against_the_oracle(device, dim, N, collider, max_steps, pe_diff_tol):
    print(f"[fire] dim={dim} N={N} {collider} max_steps={max_steps} pe_diff_tol={pe_diff_tol}", flush=True)
    st, box = packed(N, dim, seed=N, phi=0.9, ang=False)
    st.fixed[::17] = True
    ckw = dict(state=st) if collider == "CellList" else {}
    if collider == "NeighborList":
        ckw = dict(state=st, cutoff=1.2, skin=0.1, secondary_collider_type="CellList",
                   secondary_collider_kw=dict(state=st))
    mats = [jd.Material.create("elastic", density=1.0, young=1e4, poisson=0.3)]
    sy = jd.System.create(st.shape, dt=1e-3, domain_type="periodic", domain_kw=dict(box_size=box, anchor=np.zeros(dim)),
                          collider_type=collider, collider_kw=ckw, force_model_type="spring",
                          force_manager_kw=dict(gravity=np.full(dim, -3.0, np.float32)),
                          mat_table=jd.MaterialTable.from_materials(mats))
    kw = dict(max_steps=max_steps, pe_tol=0.0, pe_diff_tol=pe_diff_tol, force_tol=-1.0)
    nls = B.nl_state_of(st, sy) if collider == "NeighborList" else None
    ost = B.state_of(st)
    osteps, ope = O.minimize(ost, B.params_of(st, sy), O.FireParams(dt=float(np.float32(1e-3))), nls=nls, **kw)
    st2, _, steps, pe = jd.minimize(st, sy, **kw)
    assert steps == osteps and (pe_diff_tol < 0 or 4 < steps < max_steps)
    for f, want in (("pos_c", ost.pos), ("force", ost.force), ("torque", ost.torque)):
        assert_bitwise(f, getattr(st2, f).cpu().numpy(), want)
    assert_bitwise("q", st2.q.data.cpu().numpy(), ost.q)
    assert pe == pytest.approx(ope, rel=1e-12)


@pytest.mark.parametrize("collider", ["CellList", "NeighborList"])
@pytest.mark.parametrize("stop_at", [0, 1, 2, 3, 5, 9, 33])
def test_evaluations_past_a_stop(device, collider, stop_at):
    """A minimisation that stops by itself after a few steps: none of the
    evaluations launched past the stop with a list, whose check sees the stop,
    and otherwise none after one or two steps and fewer than half of the
    needed ones later."""
    st, box = packed(900, 3, seed=4, phi=0.9, ang=False)
    ckw = dict(state=st)
    if collider == "NeighborList":
        ckw = dict(state=st, cutoff=1.2, skin=0.1, secondary_collider_type="CellList",
                   secondary_collider_kw=dict(state=st))
    mats = [jd.Material.create("elastic", density=1.0, young=1e4, poisson=0.3)]
    sy = jd.System.create(st.shape, dt=1e-4, domain_type="periodic", domain_kw=dict(box_size=box, anchor=np.zeros(3)),
                          collider_type=collider, collider_kw=ckw, force_model_type="spring",
                          mat_table=jd.MaterialTable.from_materials(mats))
    pe = jd.minimize(st, sy, max_steps=stop_at, pe_tol=0.0, pe_diff_tol=-1.0, force_tol=-1.0)[3]
    ctx = L.context_for(device)
    ctx.set_timing(True)
    try:
        ctx.get_timing()
        st2, _, steps, _ = jd.minimize(st, sy, max_steps=1000, pe_tol=pe * (1.0 + 1e-9), pe_diff_tol=-1.0, force_tol=-1.0)
        evals = ctx.get_timing()["step_kernels"]
    finally:
        ctx.set_timing(False)
    print(f"[fire] {collider} stops at {steps}: {evals} evaluations", flush=True)
    assert steps == stop_at
    needed = steps + 1
    assert needed <= evals <= (needed if collider == "NeighborList" or steps <= 2 else needed + needed // 2)
    want = jd.minimize(st, sy, max_steps=steps, pe_tol=0.0, pe_diff_tol=-1.0, force_tol=-1.0)[0]
    assert_bitwise("force", st2.force.cpu().numpy(), want.force.cpu().numpy())
    assert_bitwise("pos", st2.pos_c.cpu().numpy(), want.pos_c.cpu().numpy())
