"""Kernels that a size selects, on both sides of the line: a system one sphere
short of it, and the same system with one more sphere that touches nothing.
The forms below the lines are held to the oracle elsewhere (traversal, list
build, float64 and precision tests); here the other form gives the same
particles the same forces, states and rows, bit for bit, since every sum is
taken in the same order."""

from __future__ import annotations

import numpy as np
import pytest

import jaxdem_amd as jd
from jaxdem_amd import precision as PR
from jaxdem_amd.utils.contacts import compute_contact_stress_tensor
from tests.test_gpu_f64 import x64
from tests.test_gpu_parity import assert_bitwise

pytestmark = pytest.mark.gpu


def one_apart(n, dim, phi, seed=1):
    """n spheres at random in a box but for a slab of its last axis, the last
    of them alone in the slab: positions, radii, velocities, box."""
    rng = np.random.Generator(np.random.PCG64(seed))
    rad = rng.uniform(0.4, 0.6, n)
    vol = (4.0 / 3.0 * np.pi * rad**3 if dim == 3 else np.pi * rad**2).sum()
    side = (vol / phi) ** (1.0 / dim)
    box = np.full(dim, side)
    pos = rng.uniform(0.7, side - 0.7, (n, dim))
    pos[:, -1] = rng.uniform(0.7, side - 5.0, n)
    pos[-1] = side / 2
    pos[-1, -1] = side - 2.5
    vel = rng.standard_normal((n, dim))
    vel[-1] = 0.0
    return pos, rad, vel, box


def system(n, dim, phi, domain, collider, law, **ckw):
    """The first n spheres of one_apart(N) for the n = N - 1 or N given as a
    pair (n, N)."""
    n, total = n
    pos, rad, vel, box = one_apart(total, dim, phi)
    mass = rad**dim
    st = jd.State.create(pos=pos[:n], rad=rad[:n], vel=vel[:n], mass=mass[:n], device="cuda")
    kw = dict(state=st, **ckw)
    mats = [jd.Material.create("elasticfrict", density=1.0, young=1e3, poisson=0.3, mu=0.4, e=0.7, mu_r=0.05)]
    sy = jd.System.create(st.shape, dt=1e-3, domain_type=domain, domain_kw=dict(box_size=box, anchor=np.zeros(dim)),
                          collider_type=collider, collider_kw=kw, force_model_type=law,
                          mat_table=jd.MaterialTable.from_materials(mats))
    return st, sy


def same(tag, a, b, n):
    assert_bitwise(tag, a.cpu().numpy()[: n - 1], b.cpu().numpy()[: n - 1])


# the first size with a lane per particle, cell edge / diameter
@pytest.mark.parametrize("f64,dim,n,edge", [
    (False, 3, 49152, 1.0), (False, 3, 98304, 0.5), (False, 2, 49152, 0.4),
    (True, 3, 32768, 1.0), (True, 2, 32768, 1.0), (True, 2, 32768, 0.4), (True, 3, 65536, 0.5),
])
@pytest.mark.parametrize("domain", ["periodic", "reflect"])
def test_cell_walk(device, f64, dim, n, edge, domain):
    print(f"[lines] walk f64={f64} dim={dim} n={n} edge={edge} {domain}", flush=True)
    out = []
    for m in (n - 1, n):
        jd.config.update("jax_enable_x64", f64)
        try:
            st, sy = system((m, n), dim, 0.6, domain, "CellList", "cundallstrack", cell_size=edge * 1.2)
            assert sy.collider.search_range == (1 if edge == 1.0 else (2 if edge == 0.5 else 3))
            f = sy.collider.compute_force(st, sy)[0]
            s2 = jd.System.step(st, sy, n=2)[0]
            e = sy.potential_energy(st)
            w = None if f64 else compute_contact_stress_tensor(st, sy)[2]
        finally:
            jd.config.update("jax_enable_x64", False)
        out.append((f, s2, e, w))
    (fa, sa, ea, wa), (fb, sb, eb, wb) = out
    assert float(fb.force[-1].abs().max()) == 0.0 and float(fa.force.abs().max()) > 0.0
    for k in ("force", "torque"):
        same(k, getattr(fa, k), getattr(fb, k), n)
    for k in ("pos_c", "vel", "ang_vel"):
        same(k, getattr(sa, k), getattr(sb, k), n)
    # float64 sums of n terms of one sign, and of 2 n contacts of both
    assert ea > 0 and abs(ea - eb) <= 1e-12 * ea
    if not f64:
        assert np.abs(wa - wb).max() <= 1e-11 * np.abs(wa).max()


@pytest.mark.parametrize("domain", ["periodic", "reflect"])
def test_list_in_work_order(device, domain):
    """A lane per sphere from 100000 on, rebuilds with live springs."""
    print(f"[lines] list {domain}", flush=True)
    out = []
    for m in (99999, 100000):
        st, sy = system((m, 100000), 3, 0.7, domain, "NeighborList", "springfriction", cutoff=1.2, skin=0.02,
                        secondary_collider_type="CellList", max_neighbors=70)
        out.append(jd.System.step(st, sy, n=12))
    (sa, ya), (sb, yb) = out
    assert ya.collider.n_build_times == yb.collider.n_build_times >= 3
    for k in ("pos_c", "vel", "ang_vel", "force", "torque"):
        same(k, getattr(sa, k), getattr(sb, k), 100000)
    assert np.array_equal(ya.collider.neighbor_list.cpu().numpy(), yb.collider.neighbor_list.cpu().numpy()[:-1])


@pytest.mark.parametrize("domain", ["periodic", "reflect"])
def test_float64_list(device, domain):
    """A lane per sphere from 131072 on."""
    print(f"[lines] float64 list {domain}", flush=True)
    out = []
    for m in (131071, 131072):
        with x64():
            st, sy = system((m, 131072), 3, 0.5, domain, "NeighborList", "hertz", cutoff=1.2, skin=0.01,
                            secondary_collider_type="CellList", max_neighbors=40)
            out.append(jd.System.step(st, sy, n=5))
    (sa, ya), (sb, yb) = out
    assert ya.collider.n_build_times == yb.collider.n_build_times >= 2
    for k in ("pos_c", "vel", "force"):
        same(k, getattr(sa, k), getattr(sb, k), 131072)
    assert np.array_equal(ya.collider.neighbor_list.cpu().numpy(), yb.collider.neighbor_list.cpu().numpy()[:-1])


@pytest.mark.parametrize("dim,skin", [(3, 0.05), (3, 1.0), (2, 0.05)])  # half-widths of one cell more and of two
def test_precise_list(device, dim, skin):
    """The precision form's list, a lane per sphere from 163840 on: positions
    and forces after a few updates (the power and energy are sums of other
    blocks, so their last bits may differ; the updates only use the sign)."""
    print(f"[lines] precise dim={dim} skin={skin}", flush=True)
    n = 163840
    pos, rad, _, box = one_apart(n, dim, 0.6)
    out = []
    for m in (n - 1, n):
        r = PR.minimize_precise(pos[:m], rad[:m], box, max_steps=4, pe_tol=0.0, pe_diff_tol=-1.0, skin=skin,
                                max_neighbors=120, device=device)
        assert r["steps"] == 4
        out.append(r)
    a, b = out
    assert float(b["force"][-1].abs().max()) == 0.0
    assert np.array_equal(a["pos"], b["pos"][:-1])
    same("force", a["force"], b["force"], n)
    assert a["pe"] * (n - 1) == pytest.approx(b["pe"] * n, rel=1e-12)
    assert np.abs(a["virial"] - b["virial"]).max() <= 1e-11 * np.abs(a["virial"]).max()
